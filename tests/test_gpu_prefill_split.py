"""GPU parity of the K-split prefill GEMM and the key-split attention (prompts of few row tiles)
with the 8-row pass path, which runs the same model through other kernels: sizes at the edges of
the 32 / 64-token tiles, of the split rules and of the change to the 128-token tiles, from slot 0
and after a cached prefix."""
import numpy as np
import pytest

from conftest import fp16_close, rel_err
from instantcua_amd import synth
from instantcua_amd.engine import Engine
from instantcua_amd.modelfile import WeightFormat

pytestmark = pytest.mark.gpu

LAYERS = 2
FMTS = {"q4": WeightFormat.Q4, "q8": WeightFormat.Q8, "f16": WeightFormat.F16}
_IMAGES = {}


def image(fmt):
    if fmt not in _IMAGES:
        _IMAGES[fmt] = synth.build_model_image(FMTS[fmt], n_layers=LAYERS, tag=f"split-{fmt}")
    return _IMAGES[fmt]


def run(e, toks, start, vis, passes, fp16=False):
    e.pass_prefill = passes
    e.prefill_fp16 = False
    if start:
        e.prefill(toks[:start], max_new=2)
    e.prefill_fp16 = fp16
    tok = e.prefill(toks[start:], start_pos=start, vis_offset=vis, max_new=2, write_logits=True)
    n = len(toks)
    return tok, e.logits(1)[0], [e.read_kv(l, k, start, n - start) for l in range(LAYERS) for k in range(2)]


def check(img, toks, start=0, vis=None):
    with Engine(flags=0, image=img, max_context=len(toks) + 8, max_steps=4) as e:
        e.eos = (-1, -1)
        off = -1
        if vis is not None:
            off = vis.vis_offset
            e.set_visual(vis.pooler.astype(np.float32), [d.astype(np.float32) for d in vis.deepstack])
            e.prepare_mrope(off, vis.llm_h, vis.llm_w)
        ref = run(e, toks, start, off, True)
        got = run(e, toks, start, off, False)
        half = run(e, toks, start, off, False, fp16=True)
    # Both paths carry ~22-bit operands and fp32 sums in another order; layer 1 reads fp16 cache
    # rows that differ by flips of their last bit (the bounds of the prefill tests).
    assert rel_err(got[1], ref[1]) < 1e-4, rel_err(got[1], ref[1])
    for i, (g, r) in enumerate(zip(got[2], ref[2])):
        if i < 2:
            fp16_close(g, r, max_ulp=1, row_tol=1e-6, frac_over_1ulp=1e-3)
        else:
            fp16_close(g, r, max_ulp=2, row_tol=2e-3, frac_over_1ulp=5e-2)
    # fp16 operands alone: 2^-12 per operand, the stated bounds of that mode.
    assert rel_err(half[1], ref[1]) < 1e-2, rel_err(half[1], ref[1])
    for g, r in zip(half[2], ref[2]):
        g, r = g.astype(np.float32), r.astype(np.float32)
        assert np.all(np.abs(g - r) <= 1e-2 * np.abs(r).max(axis=-1, keepdims=True))


@pytest.mark.parametrize("fmt", list(FMTS))
@pytest.mark.parametrize("n,start", [(9, 0), (16, 37), (32, 700), (33, 0), (64, 130), (65, 0), (129, 511), (321, 0)])
def test_split_prefill_matches_passes(fmt, n, start):
    check(image(fmt), synth.random_tokens(start + n, f"split-{n}-{start}"), start)


# hi + lo: the last size of four 64-token tiles (O and down change their width), of the K-split GEMM
# and one past each.  fp16 operands: the first sizes of the 128-token tiles of the K-split GEMM (q8
# 192, f16 320, q4 1152) and the first past it (q8 2049).  Past the K-split GEMM, where the tile of a
# product follows its count: 2000 rows (O and down on 128 x 128) and 3000 rows (QKV on 128 x 128); f16
# takes these tiles from 2049 to 2304 rows.
@pytest.mark.parametrize("fmt,n", [("q4", 256), ("q8", 257), ("q4", 1536), ("q4", 1537), ("q8", 191), ("q8", 192),
                                   ("f16", 320), ("q4", 1152), ("q8", 2049), ("q4", 2000), ("q8", 2000),
                                   ("q4", 3000), ("q8", 3000), ("f16", 2100),
                                   ("f16", 2305)])
def test_sizes_where_the_tiles_change_match_passes(fmt, n):
    check(image(fmt), synth.random_tokens(n, f"split-{n}"))


@pytest.mark.parametrize("tail", [0, 5], ids=["last-row-visual", "text-after"])
def test_split_visual_prefill_matches_passes(tail):
    """DeepStack rows are added where the down projection's partials are summed; the last layer's
    by the row that the head reads, visual or not."""
    vp = synth.visual_prompt(16 + 96 + tail, vis_offset=16, llm_h=8, llm_w=12, tag="split-vis")
    check(image("q4"), vp.tokens, 0, vp)


@pytest.mark.parametrize("n", [4192, 4300], ids=["last-row-visual", "text-after"])
def test_visual_rows_in_a_second_chunk_match_passes(n):
    """192 visual rows across the 4096-row chunks: DeepStack rows from the 97th on belong to the
    second chunk, whose down projections leave partials."""
    vp = synth.visual_prompt(n, vis_offset=4000, llm_h=12, llm_w=16, tag="split-vis2")
    check(image("q4"), vp.tokens, 0, vp)
