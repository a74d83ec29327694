"""The autotuner times the M2L's tile shapes where the batch runs on them: a
small batch in the 16-bit modes, which runs on the direct or the full-precision
kernels, leaves the plan's shape alone; one past the line has one chosen.  The
fields of either are those of the untuned plan."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["MFMA_BF16X3", "MFMA_FP16X3", "VALU"])
@pytest.mark.parametrize("K,tuned", [(1, False), (5, False), (20, True)])
def test_the_tile_shape_is_tuned_where_it_is_used(mode, K, tuned):
    import cdfmm_hip as hip

    if not hip.hip_full_available():
        pytest.skip("no gfx950 device")
    rng = np.random.default_rng(K)
    n = 9000
    x = rng.uniform(size=(n, 3))
    o = hip.UniformFmmOptions()
    o.expansion_order, o.tree.max_level = 4, 4  # 4681 boxes of 25 coefficients: 117,025 a state
    o.backend, o.precision = hip.ExecutionBackend.HIP_FULL, hip.StaticPrecision.FLOAT32
    o.hip_m2l_mode = getattr(hip.HipM2LMode, mode)
    o.fixed_target_source_indices = range(n)
    f = hip.UniformFmm(x, x, o)
    m = rng.normal(size=(K, n, 3))
    before = f.evaluate_batch(m)
    f.autotune(K)
    shape = f.hip_plan_statistics["m2l_tile_shape"]
    assert (shape != 0) == (tuned and mode != "VALU")
    np.testing.assert_array_equal(f.evaluate_batch(m), before)
