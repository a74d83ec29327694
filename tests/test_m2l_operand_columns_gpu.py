"""Columns of the tiled M2L's operands on deep trees: padded to whole tiles of 32
where the padded buffer stays within 32-bit offsets, and only there.

Depth 7, p = 4 (2,396,745 boxes): 9 states padded to 32 are 4.9 GB per half, past
the line, so the operands stay at 9 columns: the plan's memory is that of its
coefficients (2 x 35 + 2 x 25 floats) and operands (2 x 32 halves) per box and
state.  Depth 6, p = 10: 40 states padded to 64 are past it, 20 padded to 32 fit
the buffer of 40.  Fields against the FP64 plan, FP32's bar of 1e-5.
"""

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def plan(hip, x, p, depth, bits):
    o = hip.UniformFmmOptions()
    o.expansion_order, o.tree.max_level = p, depth
    o.backend = hip.ExecutionBackend.HIP_FULL
    o.precision = hip.StaticPrecision.FLOAT64 if bits == 64 else hip.StaticPrecision.FLOAT32
    o.hip_m2l_mode = hip.HipM2LMode.VALU if bits == 64 else hip.HipM2LMode.MFMA_BF16X3
    o.fixed_target_source_indices = range(len(x))
    return hip.UniformFmm(x, x, o)


@pytest.mark.parametrize("p,depth,batches", [(4, 7, (9, 20, 9)), (10, 6, (40, 20, 33))])
def test_operand_columns(p, depth, batches):
    import cdfmm_hip as hip

    if not hip.hip_full_available():
        pytest.skip("no gfx950 device")
    rng = np.random.default_rng(p)
    n = 3000
    x = rng.uniform(size=(n, 3))
    m = rng.normal(size=(max(batches), n, 3))
    states = sorted({0} | {K - 1 for K in batches})
    want = dict(zip(states, plan(hip, x, p, depth, 64).evaluate_batch(m[states])))
    f = plan(hip, x, p, depth, 32)
    base = f.hip_plan_statistics["persistent_device_bytes"]
    for i, K in enumerate(batches):
        h = f.evaluate_batch(m[:K])
        if i == 0 and depth == 7:
            boxes = (8 ** (depth + 1) - 1) // 7
            used = f.hip_plan_statistics["persistent_device_bytes"] - base
            assert used <= boxes * K * ((2 * 35 + 2 * 25) * 4 + 2 * 32 * 2) + (64 << 20)
        for k in {0, K - 1}:
            assert rel_l2(h[k], want[k]) <= 1e-5, (K, k)
        np.testing.assert_array_equal(f.evaluate_batch(m[:K]), h)
