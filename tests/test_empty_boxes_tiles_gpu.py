"""Plans of which many boxes hold no points on the tiled M2L at state counts that
are no multiple of 32: several boxes per tile (5 and 8 states), whose operands
are split for every box, and padded columns (20), in both 16-bit modes, with the
FP16 mode's small batch beside them, forward and adjoint.

As in the tests of the other state counts, against the plan of the same points
and one filler point, without a moment, in every leaf, which leaves nothing out:
relative L2 2e-6, the near field's rounding in another order.
"""

import numpy as np
import pytest

from conftest import rel_l2
from test_empty_boxes_gpu import GEOMETRIES, hip, moments, points  # noqa: F401

pytestmark = pytest.mark.gpu


def plan(hip, src, tgt, mode, p, depth):  # noqa: F811
    o = hip.UniformFmmOptions()
    o.expansion_order, o.tree.max_level = p, depth
    o.tree.root_centre = hip.Vec3(0.5, 0.5, 0.5)
    o.tree.root_half_width = 0.5
    o.backend, o.precision = hip.ExecutionBackend.HIP_FULL, hip.StaticPrecision.FLOAT32
    o.hip_m2l_mode = getattr(hip.HipM2LMode, mode)
    if src is tgt:
        o.fixed_target_source_indices = list(range(len(src)))
    return hip.UniformFmm(src, tgt, o)


@pytest.mark.parametrize("geometry", GEOMETRIES)
@pytest.mark.parametrize("mode,p,depth,batches", [("MFMA_FP16X3", 8, 4, (5, 8)), ("MFMA_BF16X3", 6, 5, (5, 8)),
                                                  ("MFMA_FP16X3", 6, 4, (1, 20)), ("MFMA_BF16X3", 4, 5, (20, 3))])
def test_outputs_are_those_of_a_plan_without_empty_boxes(hip, geometry, mode, p, depth, batches):  # noqa: F811
    src, tgt = points(geometry)
    ns, nt, side = len(src), len(tgt), 1 << depth
    fill = (np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5) / side
    filled = np.concatenate([src, fill])
    f = plan(hip, src, tgt, mode, p, depth)
    full = plan(hip, filled, filled if src is tgt else np.concatenate([tgt, fill]), mode, p, depth)
    for K in batches:  # one plan's buffers in turn
        m, c, pad = moments(ns, K, 1), moments(nt, K, 2), np.zeros((K, len(fill), 3))
        full_h = full.evaluate_batch(np.concatenate([m, pad], axis=1))[:, :nt]
        full_g = full.evaluate_adjoint_batch(np.concatenate([c, pad], axis=1))[:, :ns]
        for _ in range(2):
            assert rel_l2(f.evaluate_batch(m), full_h) <= 2e-6
            assert rel_l2(f.evaluate_adjoint_batch(c), full_g) <= 2e-6
