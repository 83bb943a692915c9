"""CPU tests of the engine's host code, against a HIP runtime of host memory (fake_hip.c).  Calls are
synchronous (icua.h): none returns with work or copies of the caller's memory pending on its stream,
and an error return in the middle of a pass does not either.  K/V ranges land where they belong in
every form of the copy."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def _run(fake, body):
    code = f"""
import ctypes as C, sys
sys.path.insert(0, {os.path.dirname(HERE)!r})
import numpy as np
from instantcua_amd import synth
from instantcua_amd.engine import Engine, EngineError
from instantcua_amd.modelfile import WeightFormat
fake = C.CDLL({fake!r})
e = Engine(flags=0, image=synth.build_model_image(WeightFormat.Q4, 1, tag="waits"), max_context=600, max_steps=4)
assert fake.fake_busy() == 0, "create"
toks = np.arange(20, dtype=np.int32)
calls = {{
    "prefill": lambda: e.prefill(toks, max_new=2, write_logits=True),
    "passes": lambda: e.prefill(toks[:5], max_new=2),
    "verify": lambda: e.verify(toks[:3]),
    "verify_logits": lambda: e.verify(toks[:3], want_logits=True),
    "set_position": lambda: e.set_position(3, 7),
    "decode": lambda: e.decode_steps(2),
    "layer_step": lambda: e.layer_step(0, np.zeros((2, 2048), np.float32), 3),
}}
{body}
print("done")
"""
    preload = ":".join(filter(None, [fake, os.environ.get("LD_PRELOAD")]))
    r = subprocess.run([sys.executable, "-c", code], env={**os.environ, "LD_PRELOAD": preload}, capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().endswith("done"), r.stdout[-2000:] + r.stderr[-2000:]


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hip") / "libfakehip.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "fake_hip.c")], check=True)
    return so


def test_calls_return_with_nothing_pending(fake):
    _run(fake, """
for name, call in calls.items():
    call()
    assert fake.fake_busy() == 0, name
""")


def test_error_returns_leave_nothing_pending(fake):
    """Every kernel launch of a call fails in turn."""
    _run(fake, """
for name, call in calls.items():
    call()
    fake.fake_arm(0)
    call()
    n = fake.fake_launches()  # (a decode has none: it replays the graph of its first call)
    for k in range(1, n + 1):
        fake.fake_arm(k)
        try:
            call()
            raise SystemExit(f"{name}: launch {k} of {n} failed unseen")
        except EngineError:
            pass
        assert fake.fake_busy() == 0, f"{name}: launch {k} of {n}"
""")


def test_kv_ranges_round_trip(fake):
    """Sizes on either side of the changes between one strided copy and a copy a group."""
    _run(fake, """
rng = np.random.default_rng(0)
for kind in (0, 1):
    full = rng.integers(0, 1 << 16, (8, 600, 128)).astype(np.uint16).view(np.float16)
    e.write_kv(0, kind, 0, full)
    for slot0, n in ((0, 600), (3, 1), (5, 64), (5, 65), (7, 511), (7, 512), (599, 1)):
        new = rng.integers(0, 1 << 16, (8, n, 128)).astype(np.uint16).view(np.float16)
        full[:, slot0:slot0 + n] = new
        e.write_kv(0, kind, slot0, new)
        assert np.array_equal(e.read_kv(0, kind, slot0, n).view(np.uint16), new.view(np.uint16)), n
        assert np.array_equal(e.read_kv(0, kind, 0, 600).view(np.uint16), full.view(np.uint16)), n
""")


def test_null_stream_work_is_waited_for(fake):
    """The engine's stream does not wait for the null stream: nothing starts on it while a clear of
    new buffers may be running there."""
    _run(fake, """
fake.fake_arm(0)
for name, call in calls.items():
    call()
    assert fake.fake_overlaps() == 0, name
e.prefill(np.arange(300, dtype=np.int32), max_new=2)
assert fake.fake_overlaps() == 0, "longer prefill"
""")


def test_prefill_buffers(fake):
    """The partials' buffer is allocated once, whatever prompts follow, and closing frees everything."""
    _run(fake, """
fake.fake_watch(C.c_size_t(4 * 256 * 128 * 256))
for n in (9, 20, 200, 400, 590):
    e.prefill(np.arange(n, dtype=np.int32), max_new=2)
    assert fake.fake_seen() == 1, n
e.close()
assert fake.fake_live() == 0, fake.fake_live()
""")
