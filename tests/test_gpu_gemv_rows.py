"""GPU parity of the multi-row products at the edges of their forms: four and five rows (the staged
forms of 4 and 8), one row block, and K = 6144 up to and past the rows that are split over three
workgroups, called twice (the arrival counters are back at zero after a call)."""
import numpy as np
import pytest

from conftest import rel_err
from instantcua_amd import engine as eng
from instantcua_amd import synth
from instantcua_amd.modelfile import WeightFormat

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [WeightFormat.Q4, WeightFormat.Q8], ids=["q4", "q8"])
@pytest.mark.parametrize("K,N", [(2048, 16), (2048, 4112), (6144, 16), (6144, 4096), (6144, 4112)])
def test_rows_and_splits_match_the_oracle(oracle_mod, fmt, K, N):
    mat = synth.make_matrix(fmt, N, K, tag="rows", index=fmt)
    tc, ts = eng.repack(fmt, eng.DeviceBuffer.from_array(mat.codes), eng.DeviceBuffer.from_array(mat.sb), N, K)
    x = np.random.default_rng(N + K).standard_normal((8, K)).astype(np.float32)
    ref = oracle_mod.gemv(fmt, mat.codes, mat.sb, N, K, x)
    xb = eng.DeviceBuffer.from_array(x)
    for m in (2, 4, 5, 8):
        for _ in range(2):
            y = eng.DeviceBuffer.from_array(np.full((m, N), np.nan, np.float32))
            eng.gemv(fmt, tc, ts, N, K, xb, m, y)
            # 22-bit operands, fp32 group sums (the bound of the standalone products' tests)
            assert rel_err(y.to_array(np.float32, (m, N)), ref[:m]) < 2e-6, m
