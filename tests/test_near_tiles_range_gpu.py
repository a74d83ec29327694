"""Near fields on bf16 tiles in batches that are no multiple of 32, at the ends of
FP32's range: moments whose low bf16 pieces would lose bits, and pairs so close
that the products' |r|^-5 overflows.  Both keep the accuracy of FP32 pairs (a few
rounding errors of 6e-8: 2e-6).
"""

import numpy as np
import pytest

from conftest import rel_l2
from test_near_lanes_gpu import hip  # noqa: F401
from test_near_tile_line_gpu import LINE, SOURCES, evaluate, expected, plan, problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("what", list(LINE))
@pytest.mark.parametrize("K", [9, 20, 41])
def test_small_moments(hip, what, K):  # noqa: F811
    # States of ordinary moments, of moments at two small scales throughout, of
    # small moments beside one ordinary source, and one without moments.
    rng = np.random.default_rng(K)
    src, tgt, ids = problem(rng, K, what)
    m = rng.normal(size=(K, SOURCES, 3))
    m[1] *= 1e-33
    m[2] *= 1e-36
    m[3] *= 1e-36
    m[3, 5] *= 1e36
    m[4] = 0.0
    m = m.astype(np.float32).astype(np.float64)
    got = evaluate(plan(hip, src, tgt, ids), m, what)
    for k in range(6):
        for key, w in expected(tgt, src, m[k], ids, what).items():
            if k == 4:
                assert not got[key][k].any()
            else:
                assert rel_l2(got[key][k] / np.abs(w).max(), w / np.abs(w).max()) <= 2e-6, k


@pytest.mark.parametrize("what", list(LINE))
@pytest.mark.parametrize("K", [9, 20, 41])
def test_close_pairs(hip, what, K):  # noqa: F811
    # A target beside each source, 2^-24 to 2^-38 of the box away (gradients: to
    # 2^-30, past which |r|^-4 leaves FP32), all coordinates exact in the two
    # FP32 parts of a position: such a target's values are one pair's.
    rng = np.random.default_rng(K)
    _, tgt, ids = problem(rng, K, what)
    src = rng.integers(1 << 17, 7 << 17, size=(SOURCES, 3)) * 2.0 ** -20
    far = 30 if what == "gradient" else 38
    away = rng.normal(size=(SOURCES, 3))
    away *= 2.0 ** -rng.uniform(24, far, size=(SOURCES, 1)) / np.linalg.norm(away, axis=1, keepdims=True)
    close = src + np.round(away * 2.0 ** 44) * 2.0 ** -44
    tgt = np.concatenate([close, tgt[SOURCES:]])
    ids = np.full(len(tgt), -1)
    m = rng.normal(size=(K, SOURCES, 3)).astype(np.float32).astype(np.float64)
    got = evaluate(plan(hip, src, tgt, ids), m, what)
    for k in sorted({0, K // 2, K - 1}):
        for key, w in expected(close, src, m[k], ids[:SOURCES], what).items():
            g = got[key][k][:SOURCES]
            if key == "phi":  # cancels in u.m: relative to |m| / (4 pi |r|^2)
                size = np.linalg.norm(m[k], axis=1) / (4 * np.pi * ((close - src) ** 2).sum(axis=1))
                assert (np.abs(g - w) / size).max() <= 2e-6
            else:
                assert (np.linalg.norm(g - w, axis=1) / np.linalg.norm(w, axis=1)).max() <= 2e-6
