"""The FP16 M2L mode on both sides of the batch size where it takes its split
operands: past it, on tiles with several boxes (2 to 8 states) and with padded
columns (9 and more), 22 bits per operand come closer to the FP32 M2L than the
bf16 mode's 16, without being it; a small batch is the plain mode's, bit for bit.
"""

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def modes(p, depth, n, K):
    import cdfmm_hip as hip

    if not hip.hip_full_available():
        pytest.skip("no gfx950 device")
    rng = np.random.default_rng(100 * p + K)
    x = rng.uniform(size=(n, 3))
    o = hip.UniformFmmOptions()
    o.expansion_order, o.tree.max_level = p, depth
    o.backend, o.precision = hip.ExecutionBackend.HIP_FULL, hip.StaticPrecision.FLOAT32
    o.fixed_target_source_indices = range(n)
    f = hip.UniformFmm(x, x, o)
    m = rng.normal(size=(K, n, 3))
    out = {}
    for mode in ("VALU", "MFMA_FP16X3", "MFMA_BF16X3"):
        f.set_m2l_mode(getattr(hip.HipM2LMode, mode))
        out[mode] = f.evaluate_batch(m)
    return out


@pytest.mark.parametrize("p,depth,n,K", [(8, 4, 30000, 6), (8, 4, 30000, 8), (8, 4, 30000, 12), (4, 5, 60000, 3),
                                         (6, 4, 30000, 31)])
def test_closer_to_full_precision_than_bf16(p, depth, n, K):
    out = modes(p, depth, n, K)
    for k in sorted({0, K // 2, K - 1}):
        d16, dbf = (rel_l2(out[mode][k], out["VALU"][k]) for mode in ("MFMA_FP16X3", "MFMA_BF16X3"))
        assert 0 < d16 < dbf <= 1e-5


@pytest.mark.parametrize("p,depth,n,K", [(8, 3, 20000, 1), (4, 3, 8000, 1), (6, 4, 30000, 7), (4, 3, 8000, 20)])
def test_a_small_batch_is_the_plain_mode(p, depth, n, K):
    out = modes(p, depth, n, K)
    np.testing.assert_array_equal(out["MFMA_FP16X3"], out["VALU"])
    assert (out["MFMA_BF16X3"] != out["VALU"]).any()
