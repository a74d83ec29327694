"""Plans of which many boxes hold no points, on the M2L that leaves them out:
uneven blobs, sources in a slab seen from a plane, a single occupied corner, and
sources and targets in opposite corners, for each M2L kernel, forward and
adjoint.

Each is compared with the plan of the same points and one filler point, without
a moment, in every leaf, which has no box to leave out.  The fillers come last
in their leaves, so multipoles, M2L and L2P are the same operations; near-field
sums are the same terms in another order: relative L2 2e-6 in FP32, 1e-13 in
FP64.  The full-precision modes are compared with the FP64 CPU restatement too
(1e-5 and 1e-12).  Locals of boxes without targets are the sources' field there
all the same: against the restatement with a target in every box.
"""

import functools

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

GEOMETRIES = ["blobs", "slab", "corner", "opposite"]


@pytest.fixture(scope="module")
def hip():
    import cdfmm_hip

    if not cdfmm_hip.hip_full_available():
        pytest.skip("no gfx950 device")
    return cdfmm_hip


def points(geometry):
    rng = np.random.default_rng(11)
    if geometry == "blobs":
        x = np.concatenate([rng.normal(c, 0.03, size=(900, 3)) for c in ([0.2, 0.3, 0.6], [0.7, 0.75, 0.3])])
        return x, x
    if geometry == "slab":
        src = rng.uniform([0, 0, 0.05], [1, 1, 0.15], size=(2000, 3))
        return src, np.concatenate([rng.uniform(0, 1, size=(700, 2)), np.full((700, 1), 0.55)], axis=1)
    if geometry == "corner":
        x = rng.uniform(0, 0.24, size=(1500, 3))
        return x, x
    return rng.uniform(0, 0.3, size=(1200, 3)), rng.uniform(0.7, 1, size=(900, 3))


def plan(hip, src, tgt, bits, mode="VALU", p=6):
    o = hip.UniformFmmOptions()
    o.expansion_order = p
    o.tree.max_level = 4
    o.tree.root_centre = hip.Vec3(0.5, 0.5, 0.5)
    o.tree.root_half_width = 0.5
    o.backend = hip.ExecutionBackend.HIP_FULL
    o.precision = hip.StaticPrecision.FLOAT64 if bits == 64 else hip.StaticPrecision.FLOAT32
    o.hip_m2l_mode = getattr(hip.HipM2LMode, mode)
    if src is tgt:
        o.fixed_target_source_indices = list(range(len(src)))
    return hip.UniformFmm(src, tgt, o)


FILL = (np.stack(np.meshgrid(*[np.arange(16)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5) / 16
ROOT = {"root_centre": (0.5, 0.5, 0.5), "root_half_width": 0.5}


def moments(count, states, salt):
    return np.stack([np.random.default_rng(1000 * salt + k).normal(size=(count, 3)) for k in range(states)])


@functools.lru_cache(maxsize=None)
def reference(geometry, state, adjoint):
    import oracle

    src, tgt = points(geometry)
    a, b = (tgt, src) if adjoint else (src, tgt)
    ids = np.arange(len(src)) if src is tgt else None
    m = moments(len(a), state + 1, 2 if adjoint else 1)[state]
    return oracle.CpuFmm(a, b, 6, 4, 64, fixed_ids=ids, **ROOT).evaluate(m)["H"]


@pytest.mark.parametrize("geometry", GEOMETRIES)
@pytest.mark.parametrize("bits,mode,K", [(64, "VALU", 1), (64, "VALU", 5), (32, "VALU", 1), (32, "VALU", 5), (32, "VALU", 32),
                                         (32, "MFMA_BF16X3", 1), (32, "MFMA_BF16X3", 20), (32, "MFMA_BF16X3", 32),
                                         (32, "MFMA_BF16X3", 64), (32, "MFMA_FP16X3", 32)])
def test_outputs_are_those_of_a_plan_without_empty_boxes(hip, geometry, bits, mode, K):
    src, tgt = points(geometry)
    f = plan(hip, src, tgt, bits, mode)
    ns, nt = len(src), len(tgt)
    filled = np.concatenate([src, FILL])
    full = plan(hip, filled, filled if src is tgt else np.concatenate([tgt, FILL]), bits, mode)
    m, c = moments(ns, K, 1), moments(nt, K, 2)
    pad = np.zeros((K, len(FILL), 3))
    full_h = full.evaluate_batch(np.concatenate([m, pad], axis=1))[:, :nt]
    full_g = full.evaluate_adjoint_batch(np.concatenate([c, pad], axis=1))[:, :ns]
    for _ in range(2):  # forward and adjoint in turn, on the same buffers
        h, g = f.evaluate_batch(m), f.evaluate_adjoint_batch(c)
        assert rel_l2(h, full_h) <= (1e-13 if bits == 64 else 2e-6)
        assert rel_l2(g, full_g) <= (1e-13 if bits == 64 else 2e-6)
        for k in {0, K - 1} if mode == "VALU" else ():
            bar = 1e-12 if bits == 64 else 1e-5
            assert rel_l2(h[k], reference(geometry, k, False)) <= bar
            assert rel_l2(g[k], reference(geometry, k, True)) <= bar


@pytest.mark.parametrize("geometry", GEOMETRIES)
@pytest.mark.parametrize("bits,mode,K", [(64, "VALU", 1), (32, "VALU", 1), (32, "MFMA_BF16X3", 1), (32, "MFMA_BF16X3", 32)])
def test_locals_of_boxes_without_targets(hip, geometry, bits, mode, K):
    import oracle

    src, tgt = points(geometry)
    m = moments(len(src), K, 1)
    f = plan(hip, src, tgt, bits, mode, 4)
    f.evaluate_batch(m)
    full = oracle.CpuFmm(src, FILL, 4, 4, bits, **ROOT)
    full.evaluate(m[K - 1])
    # Sums over the list with cancellation, relative to the node's largest.
    bar = 1e-11 if bits == 64 else 1e-4
    for node in range(585, 585 + 4096, 61):
        want = full.coefficients("local", node)
        np.testing.assert_allclose(f.local(node, K - 1), want, rtol=0, atol=bar * np.abs(want).max())
