"""FP32 near fields of batches that are no multiple of 32 on both sides of the
number of target tiles from which they run on bf16 matrix tiles: many targets
and a quarter of them, with the same sources.

Depth 1 trees have no far field, so the outputs are the near field, and the FP64
direct sums over all pairs are their values (a few rounding errors of 6e-8 per
pair: 2e-6 relative L2).  One kernel gives a target the same bits whatever the
others are, so results that differ show that the two sides are two kernels.
"""

import numpy as np
import pytest

from conftest import rel_l2
from test_near_lanes_gpu import direct, gradient, hip  # noqa: F401

pytestmark = pytest.mark.gpu

SOURCES = 61
# tiles x states per launch where the line lies on trees of 8 leaves, by output
LINE = {"field": 15000, "both": 5500, "gradient": 7000}


def plan(hip, src, tgt, ids):  # noqa: F811
    o = hip.UniformFmmOptions()
    o.expansion_order = 2
    o.tree.max_level = 1
    o.tree.root_centre = hip.Vec3(0.5, 0.5, 0.5)  # the same box for either number of targets
    o.tree.root_half_width = 0.5
    o.backend = hip.ExecutionBackend.HIP_FULL
    o.precision = hip.StaticPrecision.FLOAT32
    o.fixed_target_source_indices = list(ids)
    return hip.UniformFmm(src, tgt, o)


def launches(K):
    return (1 if K // 32 + (K % 32 > 16) > 0 else 0) + (1 if 0 < K % 32 <= 16 else 0)


def problem(rng, K, what):
    """Sources, and targets past the line of which the first are the sources."""
    n = 16 * (LINE[what] * launches(K) // K + 1)
    src = rng.uniform(0, 1, size=(SOURCES, 3))
    tgt = np.concatenate([src, rng.uniform(0, 1, size=(n, 3))])
    ids = np.full(len(tgt), -1)
    ids[:SOURCES] = np.arange(SOURCES)
    return src, tgt, ids


def evaluate(f, m, what):
    if what == "field":
        return {"H": f.evaluate_batch(m)}
    if what == "both":
        return f.evaluate_batch_outputs(m, output="both")
    return {"G": f.evaluate_field_gradient_batch(m)}


def expected(tgt, src, m, ids, what):
    if what == "gradient":
        return {"G": gradient(tgt, src, m, ids)}
    h, phi = direct(tgt, src, m, ids)
    return {"H": h, "phi": phi} if what == "both" else {"H": h}


@pytest.mark.parametrize("what,K", [(w, K) for w in LINE for K in (9, 15, 16, 17, 31, 33, 48, 49, 63)]
                         + [("gradient", 7), ("gradient", 8)])
def test_both_sides_of_the_line(hip, what, K):  # noqa: F811
    rng = np.random.default_rng(K)
    src, tgt, ids = problem(rng, K, what)
    few = len(tgt) // 4
    m = rng.normal(size=(K, SOURCES, 3))
    many_out = evaluate(plan(hip, src, tgt, ids), m, what)
    few_out = evaluate(plan(hip, src, tgt[:few], ids[:few]), m, what)
    for k in sorted({0, K // 2, K - 1}):
        want = expected(tgt, src, m[k], ids, what)
        for key, w in want.items():
            assert rel_l2(many_out[key][k], w) <= 2e-6
            assert rel_l2(few_out[key][k], w[:few]) <= 2e-6
    assert any((many_out[key][:, :few] != few_out[key]).any() for key in many_out)


@pytest.mark.parametrize("what", list(LINE))
@pytest.mark.parametrize("K", [9, 20, 41])
def test_own_source_past_the_line_is_left_out_whatever_its_moment(hip, what, K):  # noqa: F811
    # On the tiles a target's own source has weight zero, and zero times a
    # moment that is not finite is NaN: those sums are formed again without it.
    rng = np.random.default_rng(K)
    src, tgt, ids = problem(rng, K, what)
    m = rng.normal(size=(K, SOURCES, 3))
    clean = m.copy()
    m[K - 2, 11] = [np.nan, np.inf, 1.0]
    got = evaluate(plan(hip, src, tgt, ids), m, what)
    for k in sorted({0, K - 3, K - 2, K - 1}):
        want = expected(tgt, src, clean[k], ids, what)
        for key, w in want.items():
            if k != K - 2:
                assert rel_l2(got[key][k], w) <= 2e-6
                continue
            assert rel_l2(got[key][k][11], w[11]) <= 2e-6
            others = np.arange(len(tgt)) != 11
            assert np.isnan(got[key][k].reshape(len(tgt), -1)[others]).any(axis=1).all()
