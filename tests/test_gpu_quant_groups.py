"""GPU parity of the q4 quantiser at the edges of its work split (five lanes per 64-group, twelve
groups per wavefront, four wavefronts per workgroup): one group, and counts just below, at and
above a wavefront's and a workgroup's share; and the counts where one lane per group takes over."""
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
