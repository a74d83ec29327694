"""The vector-ALU near field at the edges of its tiling: every number of states
per workgroup and across workgroups, leaves from empty to more targets than one
pass of a workgroup holds, and an identity map whose own source is not finite.

Depth 0 and 1 trees have no far field, so the outputs are the near field, and
the FP64 direct sums over all pairs are their values.  FP32 pairs carry a few
rounding errors of 6e-8 each and cancel over the sum: bar 2e-6 relative L2;
FP64 the same with 1.1e-16: bar 1e-13.
"""

import numpy as np
import pytest

from conftest import direct_field_gradient, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import cdfmm_hip

    if not cdfmm_hip.hip_full_available():
        pytest.skip("no gfx950 device")
    return cdfmm_hip


def plan(hip, src, tgt, depth, bits, ids=None):
    o = hip.UniformFmmOptions()
    o.expansion_order = 2
    o.tree.max_level = depth
    o.backend = hip.ExecutionBackend.HIP_FULL
    o.precision = hip.StaticPrecision.FLOAT64 if bits == 64 else hip.StaticPrecision.FLOAT32
    if ids is not None:
        o.fixed_target_source_indices = list(ids)
    return hip.UniformFmm(src, tgt, o)


def direct(tgt, src, m, ids):
    """Fields and potentials of all pairs but each target's own source."""
    r = tgt[:, None, :] - src[None, :, :]
    d = np.linalg.norm(r, axis=2)
    if ids is not None:
        own = ids >= 0
        d[np.flatnonzero(own), ids[own]] = np.inf
    mr = np.einsum("tsc,sc->ts", r, m)
    f = 1.0 / (4.0 * np.pi * d ** 3)
    h = np.einsum("ts,tsc->tc", 3.0 * f * mr / d ** 2, r) - f @ m
    return h, (f * mr).sum(axis=1)


def points(rng, n):
    """n points of which most lie in one octant, one octant holding a single
    point and one none."""
    x = rng.uniform(0.0, 0.5, size=(n, 3))
    x[1::7] += [0.5, 0.0, 0.0]
    x[2::13] += [0.0, 0.5, 0.5]
    x[0] = [0.9, 0.9, 0.9]
    x[3] = [0.0, 0.9, 0.1]
    return x


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("depth", [0, 1])
@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 6, 7, 8, 9, 17, 33])
def test_every_state_count_against_the_direct_sum(hip, bits, depth, K):
    rng = np.random.default_rng(100 * K + depth)
    x = points(rng, 301)
    ids = np.arange(301)
    ids[5:20:3] = -1  # a target there sits on a source only if the map says so
    tgt = x.copy()
    tgt[ids < 0] += 0.011
    m = rng.normal(size=(K, 301, 3))
    f = plan(hip, x, tgt, depth, bits, ids)
    bar = 2e-6 if bits == 32 else 1e-13
    h = f.evaluate_batch(m)
    both = f.evaluate_batch_outputs(m, output="both")
    g = f.evaluate_field_gradient_batch(m)
    for k in sorted({0, K // 2, K - 1}):
        want, phi = direct(tgt, x, m[k], ids)
        assert rel_l2(h[k], want) <= bar
        assert rel_l2(both["H"][k], want) <= bar
        assert rel_l2(both["phi"][k], phi) <= bar
        assert rel_l2(g[k], gradient(tgt, x, m[k], ids)) <= bar


def gradient(tgt, src, m, ids):
    """direct_field_gradient with targets without an own source (-1) too."""
    out = np.empty((len(tgt), 6))
    own = ids >= 0
    out[own] = direct_field_gradient(tgt[own], src, m, ids[own])
    out[~own] = direct_field_gradient(tgt[~own], src, m)
    return out


@pytest.mark.parametrize("bits", [32, 64])
def test_own_source_is_left_out_whatever_its_moment(hip, bits):
    # A target's own source is skipped, not multiplied by zero.
    rng = np.random.default_rng(7)
    x = points(rng, 90)
    m = rng.normal(size=(90, 3))
    want, _ = direct(x, x, m, np.arange(90))
    m[11] = [np.nan, np.inf, 1.0]
    h = plan(hip, x, x, 1, bits, range(90)).evaluate(m)["H"]
    assert rel_l2(h[11], want[11]) <= (2e-6 if bits == 32 else 1e-13)
    assert np.isnan(h[np.arange(90) != 11]).any(axis=1).all()
