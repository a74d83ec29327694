"""Locals of boxes without targets are formed once per evaluate, when the first
of them is read, and again after the next evaluate.

How often shows in the runtime calls of a read: a copy takes six checked calls,
the M2L and the downward pass of a depth 4 tree five more, so an error armed
behind eight meets only a read that forms the locals.
"""

import ctypes
import os

import numpy as np
import pytest

from conftest import REPO
from test_empty_boxes_gpu import hip, moments, plan, points  # noqa: F401

pytestmark = pytest.mark.gpu

HIP_ERROR_LAUNCH_FAILURE = 719


@pytest.mark.parametrize("bits,mode,K", [(64, "VALU", 1), (32, "VALU", 1), (32, "MFMA_BF16X3", 5), (32, "MFMA_BF16X3", 32)])
def test_reads_after_the_first_are_copies(hip, bits, mode, K):  # noqa: F811
    lib = ctypes.CDLL(os.path.join(REPO, "dip-fmm_amd", "libhipfmm.so"))
    lib.hipfmm_debug_inject_error.argtypes = [ctypes.c_int, ctypes.c_int]
    src, tgt = points("opposite")
    f = plan(hip, src, tgt, bits, mode, 4)
    nodes = [585, 585 + 7, 585 + 100]  # leaves of the sources' corner, where no targets are

    def forms_locals(node):
        lib.hipfmm_debug_inject_error(HIP_ERROR_LAUNCH_FAILURE, 8)
        try:
            f.local(node, K - 1)
            return False
        except RuntimeError:
            return True
        finally:
            lib.hipfmm_debug_inject_error(0, 0)

    for salt in (1, 2):
        f.evaluate_batch(moments(len(src), K, salt))
        assert forms_locals(nodes[0])
        first = [np.array(f.local(node, K - 1)) for node in nodes]
        assert not any(forms_locals(node) for node in nodes)
        for node, want in zip(nodes, first):
            np.testing.assert_array_equal(f.local(node, K - 1), want)
        fresh = plan(hip, src, tgt, bits, mode, 4)  # the same locals from a plan of its own
        fresh.evaluate_batch(moments(len(src), K, salt))
        for node, want in zip(nodes, first):
            np.testing.assert_array_equal(fresh.local(node, K - 1), want)
            assert np.abs(want).max() > 0
