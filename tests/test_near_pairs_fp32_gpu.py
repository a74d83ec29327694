"""Single FP32 near-field pairs, each target with one source (a depth 0 tree has
no far field), where the arithmetic of a pair shows: its constant factors.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def plan(src, tgt):
    import cdfmm_hip as hip

    if not hip.hip_full_available():
        pytest.skip("no gfx950 device")
    o = hip.UniformFmmOptions()
    o.expansion_order = 2
    o.tree.max_level = 0
    o.tree.root_centre = hip.Vec3(0.5, 0.5, 0.5)
    o.tree.root_half_width = 0.5
    o.backend = hip.ExecutionBackend.HIP_FULL
    o.precision = hip.StaticPrecision.FLOAT32
    return hip.UniformFmm(src, tgt, o)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("K", [1, 2, 3, 8])
def test_the_axial_field_is_twice_the_transverse(axis, K):
    # H = f (3 (u.m) u - m).  At a power of two along an axis every factor but f
    # is exact (the hardware root of a power of four is), so the field of a
    # moment along the axis is exactly 2 f and that of one across it -f: any
    # rounding of the 3 shows as a different ratio.
    src = np.array([[0.25, 0.25, 0.25]])
    tgt = np.repeat(src, 20, axis=0)
    tgt[:, axis] += 0.5 ** np.arange(1, 21)
    f = plan(src, tgt)
    across = (axis + 1) % 3
    fields = {}
    for c in (axis, across):
        m = np.zeros((K, 1, 3))
        m[:, 0, c] = 1.0
        for outputs in (f.evaluate_batch(m), f.evaluate_batch_outputs(m, output="both")["H"]):
            fields.setdefault(c, []).append(np.asarray(outputs)[:, :, c])
    for a, b in zip(fields[axis], fields[across]):
        assert (b < 0).all()
        np.testing.assert_array_equal(a, -2.0 * b)


@pytest.mark.parametrize("K", [1, 3, 8])
def test_pairs_have_no_common_error(K):
    # Roundings average out over many pairs; a factor that is off does not.  The
    # hardware root is 0.7e-8 short on average, thrice in f and once more in each
    # u of 3 (u.m) u: some 4e-8 of the field, and the roundings' mean over 20,000
    # targets 1e-9.  One more factor rounded with one sign (1 / (4 pi): 4e-8) is
    # past 7e-8.
    rng = np.random.default_rng(K)
    src = np.array([[0.45, 0.55, 0.5]])
    tgt = rng.uniform(0, 1, size=(20000, 3))
    m = rng.normal(size=(K, 1, 3)).astype(np.float32).astype(np.float64)
    f = plan(src, tgt)
    r = tgt - src
    n = np.linalg.norm(r, axis=1, keepdims=True)
    u = r / n
    for h in (f.evaluate_batch(m), f.evaluate_batch_outputs(m, output="both")["H"]):
        for k in range(K):
            want = (3.0 * (u * m[k]).sum(axis=1, keepdims=True) * u - m[k]) / (4.0 * np.pi * n ** 3)
            off = ((h[k] - want) * want).sum(axis=1) / (want ** 2).sum(axis=1)
            assert abs(off.mean()) <= 7e-8
