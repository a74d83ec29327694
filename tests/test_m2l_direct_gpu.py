"""The M2L that works without staged operands: every order (row tiles, the last
row apart, part-filled depth groups), every way the offsets are shared over the
waves of a workgroup (1, 2, 4, 8 and 16, by the number of columns), both
coefficient layouts (states in runs; K a multiple of 32 interleaved), and the
16-bit modes on either side of the batch size where they leave it.

Bars: FP64 1e-12 against the oracle's FP64 FMM; the FP32 modes 1e-5 against
the same.  A repeated evaluate is bitwise the first.
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


def check(hip, oracle_mod, p, depth, n, batches):
    rng = np.random.default_rng(100 * p + depth)
    x = rng.uniform(0.0, 1.0, size=(n, 3))
    x[: n // 4] = 0.3 * x[: n // 4] ** 2  # denser near one corner of the grid
    ids = np.arange(n)
    ref = oracle_mod.CpuFmm(x, x, p, depth, 64, fixed_ids=ids)
    m = rng.normal(size=(max(batches), n, 3))
    want = {k: ref.evaluate(m[k], ids)["H"] for k in {0} | {K - 1 for K in batches}}

    def plan(bits):
        o = hip.UniformFmmOptions()
        o.expansion_order = p
        o.tree.max_level = depth
        o.backend = hip.ExecutionBackend.HIP_FULL
        o.precision = hip.StaticPrecision.FLOAT64 if bits == 64 else hip.StaticPrecision.FLOAT32
        o.fixed_target_source_indices = list(ids)
        return hip.UniformFmm(x, x, o)

    f64, f32 = plan(64), plan(32)
    for K in batches:
        h = f64.evaluate_batch(m[:K])
        for k in {0, K - 1}:
            assert rel_l2(h[k], want[k]) <= 1e-12
        for mode in ("VALU", "MFMA_BF16X3", "MFMA_FP16X3"):
            f32.set_m2l_mode(getattr(hip.HipM2LMode, mode))
            h = f32.evaluate_batch(m[:K])
            for k in {0, K - 1}:
                assert rel_l2(h[k], want[k]) <= 1e-5, (mode, K, k)
            np.testing.assert_array_equal(f32.evaluate_batch(m[:K]), h)


@pytest.mark.parametrize("p", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10])
def test_every_order(hip, oracle_mod, p):
    check(hip, oracle_mod, p, 3, 700, (1, 3, 32))


@pytest.mark.parametrize("p,depth,batches", [(2, 5, (1, 2, 4, 8)), (6, 4, (1, 9, 14, 16, 40)), (4, 2, (1, 2, 33))])
def test_every_share_of_the_offsets(hip, oracle_mod, p, depth, batches):
    check(hip, oracle_mod, p, depth, 2000, batches)
