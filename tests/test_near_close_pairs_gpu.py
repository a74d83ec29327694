"""FP64 near-field pairs from 1e-12 of the box apart to across it: the reciprocal
square root holds its precision at every exponent, and a coincident pair that is
no identity pair gives NaN.

Each target has one source, so its field is one pair's: some 20 roundings of
1.1e-16, a few of them amplified by the cancellation in 3 (u.m) u - m (at most
4 |m| against at least |m|): bar 1e-14 of the field's norm.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 4, 5])
def test_fp64_pairs_of_every_distance(K):
    import cdfmm_hip as hip

    if not hip.hip_full_available():
        pytest.skip("no gfx950 device")
    rng = np.random.default_rng(K)
    src = np.array([[0.25, 0.5, 0.75]])
    u = rng.normal(size=(240, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    tgt = src + u * np.logspace(-12, -0.7, 240)[:, None]
    tgt[0] = src[0]
    o = hip.UniformFmmOptions()
    o.expansion_order = 2
    o.tree.max_level = 0
    o.backend = hip.ExecutionBackend.HIP_FULL
    o.precision = hip.StaticPrecision.FLOAT64
    m = rng.normal(size=(K, 1, 3))
    r = hip.UniformFmm(src, tgt, o).evaluate_batch_outputs(m, output="both")
    d = tgt - src
    with np.errstate(all="ignore"):
        n = np.linalg.norm(d, axis=1, keepdims=True)
        e = d / n
        for k in range(K):
            em = (e * m[k]).sum(axis=1, keepdims=True)
            h, phi = (3.0 * em * e - m[k]) / (4.0 * np.pi * n ** 3), em[:, 0] / (4.0 * np.pi * n[:, 0] ** 2)
            assert np.isnan(r["H"][k][0]).all() and np.isnan(r["phi"][k][0])
            err = np.linalg.norm(r["H"][k] - h, axis=1) / np.linalg.norm(h, axis=1)
            assert err[1:].max() <= 1e-14
            # the potential's own cancellation is that of e.m
            scale = np.linalg.norm(m[k]) / (4.0 * np.pi * n[:, 0] ** 2)
            assert (np.abs(r["phi"][k] - phi) / scale)[1:].max() <= 1e-14
