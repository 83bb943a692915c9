"""GPU parity of the q4 quantiser at the edges of its work split (five lanes per 64-group, twelve
groups per wavefront, four wavefronts per workgroup): one group, and counts just below, at and
above a wavefront's and a workgroup's share; and the counts where one lane per group takes over.
And of its rounding (one conversion where the reference rounds halves away from zero) where the
nearest wrong rounding would change bytes."""
import numpy as np
import pytest

from instantcua_amd import convert

from test_gpu_quant import edge_matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups", [1, 11, 12, 13, 47, 48, 49, 97, 131071, 131103])
def test_q4_group_counts_match_the_oracle(oracle_mod, groups):
    m = edge_matrix(1, 64 * groups, seed=groups)
    c, s = convert.quantize_q4_raw(m)
    rc, rs = oracle_mod.quant_q4(m)
    assert np.array_equal(s, rs) and np.array_equal(c, rc)


# Groups w = s (q - offset), as (s, offset, 2 q in base 32).  In the first six, halves times the
# reciprocal of the fitted scale come out one ulp below 1/2: they round to 0, and floor(x + 1/2) in
# float32 gives 1.  The others hold ties k + 1/2 with k = 0, 2, .. 14, which round up, to even down.  With
# either wrong rounding the oracle gives other bytes.
ROUNDING = [
    ("0x1.6dc000p-8", 15, "0u1uuu00u00u00u0u0u000uuuuuuu0u00u0uuu0u000u000000uuu0u0uu000u00"),
    ("0x1.6dc000p-4", 7, "0u1u0u00u0u000uuu0u00u00uuuu000u00000uuuuu0000uu00uuuuu0u00u0u00"),
    ("0x1.44c000p-8", 10, "0u1u0uuuu0u0uu00u0uuu0uuu00u00uu0uu0uu0uu00u00u00000u000uuuuuuuu"),
    ("0x1.24c000p-5", 4, "0u1s2s004qqsuu4222ss4q04042uq0squ04u04404uuss4uuusuu004420224440"),
    ("0x1.4c0000p-6", 8, "0u1ff0000uu0u000000000000000u00u0u00u0u00uu0u000uuu0u0u0uuuu00u0"),
    ("0x1.8bc000p-8", 13, "0u1qu4qq2q0suq4us42uq2s2qs4s2u424002q04s2u2q0s2susq0u0us2qq0s42q"),
    ("0x1.450000p-6", 11, "0ut1u0u00uu0uuuuu0uu0uu0uuu000uu0000u0uuu0000u000uu0u000uu00uuuu"),
    ("0x1.158000p-5", 12, "0u5hp00uu0u0uu0uuu0uuu000u000000uu0u0uu000u0000uuuuuu00u0uuu0u00"),
    ("0x1.024000p-7", 4, "0u9uuu0000u00uuuu0uuu0u00u000u0u0u0uu0uu0u0uu0000u0u000000uuuu0u"),
    ("0x1.370000p-7", 7, "0ud8qso4ga0kc8e2k06caa2c6gg2iui2o8cqam6ccugkgsoc0gui08aee4u6e6kk"),
    ("0x1.e18000p-6", 8, "0uh0u0uuu0u0u00u0u00u0uu0uuuuu00uuuuuu00uu0uuu0uuuuuuuuu0uu00000"),
    ("0x1.14c000p-5", 8, "0uls04qs4quus0uqsu2usqqs40su24sq4qqq2ssuqs00us0q24qqs0s40u4004uu"),
    ("0x1.158000p-5", 12, "0u5hp00uu0u0uu0uuu0uuu000u000000uu0u0uu000u0000uuuuuu00u0uuu0u00"),
    ("0x1.450000p-6", 11, "0ut1u0u00uu0uuuuu0uu0uu0uuu000uu0000u0uuu0000u000uu0u000uu00uuuu"),
]


def rounding_matrix():
    rows = []
    for s, off, codes in ROUNDING:
        s = np.float32(float.fromhex(s))
        rows.append(-s * np.float32(off) + s * np.array([int(c, 32) / 2 for c in codes], np.float32))
    return np.stack(rows).astype(np.float32)


def test_q4_rounding_matches_the_oracle_next_to_halves(oracle_mod):
    m = rounding_matrix()
    rc, rs = oracle_mod.quant_q4(m)
    c, s = convert.quantize_q4_raw(m)
    assert np.array_equal(s, rs) and np.array_equal(c, rc)
    big = np.tile(m, (131072 // len(m) + 1, 1))  # one lane a group instead of five
    c, s = convert.quantize_q4_raw(big)
    assert np.array_equal(s, np.resize(rs, s.shape)) and np.array_equal(c, np.resize(rc, c.shape))
