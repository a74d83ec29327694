"""The far-field kernels for any number of states at the edges of their tiles:
orders whose coefficients leave part-filled row tiles and last depth batches,
state counts that leave part-filled column tiles, fill exactly four, or start
another chunk (fields 21 / 22, potentials 16 / 17, gradients 10 / 11), empty
leaves, and trees from two levels up.

Against the oracle's FP64 FMM of the same order and tree: FP64 to 1e-12, FP32
to 1e-5 (the bars of the two precisions); field gradients against the FP64
plan's, whose values the gradient tests pin.
"""

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import cdfmm_hip

    if not cdfmm_hip.hip_full_available():
        pytest.skip("no gfx950 device")
    return cdfmm_hip


def plan(hip, x, p, depth, bits, mode="VALU"):
    o = hip.UniformFmmOptions()
    o.expansion_order = p
    o.tree.max_level = depth
    o.backend = hip.ExecutionBackend.HIP_FULL
    o.precision = hip.StaticPrecision.FLOAT64 if bits == 64 else hip.StaticPrecision.FLOAT32
    o.hip_m2l_mode = getattr(hip.HipM2LMode, mode)
    o.fixed_target_source_indices = list(range(len(x)))
    return hip.UniformFmm(x, x, o)


def points(rng, n):
    """Two clusters and a thin background: most leaves of depth 3 are empty."""
    x = rng.uniform(0.0, 1.0, size=(n, 3))
    x[: n // 3] = 0.1 + 0.05 * rng.standard_normal((n // 3, 3)).clip(-1.9, 1.9)
    x[n // 3 : n // 2, 2] *= 0.2
    return x


@pytest.mark.parametrize("p,depth", [(1, 2), (2, 3), (4, 2), (5, 4), (7, 3), (8, 3), (9, 3), (10, 2)])
@pytest.mark.parametrize("K", [1, 2, 5, 16, 17, 21, 22, 43])
def test_every_order_and_state_count_against_the_oracle(hip, oracle_mod, p, depth, K):
    rng = np.random.default_rng(1000 * p + K)
    n = 501
    x = points(rng, n)
    ids = np.arange(n)
    m = rng.normal(size=(K, n, 3))
    ref = oracle_mod.CpuFmm(x, x, p, depth, 64, fixed_ids=ids)
    states = sorted({0, K // 2, K - 1})
    want = {k: ref.evaluate(m[k], ids, output="both") for k in states}
    f64 = plan(hip, x, p, depth, 64)
    g64 = f64.evaluate_field_gradient_batch(m)
    for bits, bar in ((64, 1e-12), (32, 1e-5)):
        f = f64 if bits == 64 else plan(hip, x, p, depth, 32, "MFMA_BF16X3" if p >= 2 else "VALU")
        h = f.evaluate_batch(m)
        both = f.evaluate_batch_outputs(m, output="both")
        only = f.evaluate_batch_outputs(m, output="potential")
        g = f.evaluate_field_gradient_batch(m)
        assert only["H"] is None
        for k in states:
            assert rel_l2(h[k], want[k]["H"]) <= bar
            assert rel_l2(both["H"][k], want[k]["H"]) <= bar
            assert rel_l2(both["phi"][k], want[k]["phi"]) <= bar
            assert rel_l2(only["phi"][k], want[k]["phi"]) <= bar
            assert rel_l2(g[k], g64[k]) <= bar
