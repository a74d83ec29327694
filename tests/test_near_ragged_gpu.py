"""FP32 near fields on the matrix cores for batches that are no multiple of 32:
the state counts around the 16- and 32-state tiles and around the counts where
the vector ALUs hand over, and an own source that is not finite.

Depth 0 and 1 trees have no far field, so the outputs are the near field, and
the FP64 direct sums over all pairs are their values (the bars of the
vector-ALU near field: a few rounding errors of 6e-8 per pair, 2e-6 relative
L2).
"""

import numpy as np
import pytest

from conftest import rel_l2
from test_near_lanes_gpu import direct, gradient, hip, plan, points  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [6, 7, 8, 9, 15, 16, 17, 31, 33, 47, 48, 49, 63])
def test_state_tiles_against_the_direct_sum(hip, K):  # noqa: F811
    rng = np.random.default_rng(K)
    x = points(rng, 131)
    ids = np.arange(131)
    m = rng.normal(size=(K, 131, 3))
    f = plan(hip, x, x, 1, 32, ids)
    h = f.evaluate_batch(m)
    both = f.evaluate_batch_outputs(m, output="both")
    g = f.evaluate_field_gradient_batch(m)
    for k in range(K):
        want, phi = direct(x, x, m[k], ids)
        assert rel_l2(h[k], want) <= 2e-6
        assert rel_l2(both["H"][k], want) <= 2e-6
        assert rel_l2(both["phi"][k], phi) <= 2e-6
        assert rel_l2(g[k], gradient(x, x, m[k], ids)) <= 2e-6


@pytest.mark.parametrize("K", [9, 20, 41])
def test_own_source_is_left_out_whatever_its_moment(hip, K):  # noqa: F811
    # A target's own source is skipped, not multiplied by zero; the states
    # whose moments are all finite keep their values.
    rng = np.random.default_rng(K)
    x = points(rng, 90)
    ids = np.arange(90)
    m = rng.normal(size=(K, 90, 3))
    clean = m.copy()
    m[K - 2, 11] = [np.nan, np.inf, 1.0]
    f = plan(hip, x, x, 1, 32, ids)
    h = f.evaluate_batch(m)
    g = f.evaluate_field_gradient_batch(m)
    for k in range(K):
        want, _ = direct(x, x, clean[k], ids)
        dwant = gradient(x, x, clean[k], ids)
        if k == K - 2:
            assert rel_l2(h[k][11], want[11]) <= 2e-6 and rel_l2(g[k][11], dwant[11]) <= 2e-6
            others = np.arange(90) != 11
            assert np.isnan(h[k][others]).any(axis=1).all() and np.isnan(g[k][others]).any(axis=1).all()
        else:
            assert rel_l2(h[k], want) <= 2e-6 and rel_l2(g[k], dwant) <= 2e-6
