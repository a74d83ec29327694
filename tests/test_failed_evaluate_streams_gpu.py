"""An evaluate that fails half-way on one stream, and the next one on another.

Its kernels work on the plan's buffers, so they have ended when the error is
reported: an evaluate that follows at once on another stream, from host memory
or in a group gives the plan's own results bit for bit.
"""

import ctypes
import os

import numpy as np
import pytest

from conftest import REPO

pytestmark = pytest.mark.gpu

HIP_ERROR_LAUNCH_FAILURE = 719


@pytest.mark.parametrize("bits,K,mode", [(32, 32, "MFMA_BF16X3"), (32, 5, "VALU"), (64, 2, "VALU")])
def test_the_next_evaluate_after_a_failure(bits, K, mode):
    import cdfmm_hip as hip
    import torch

    if not hip.hip_full_available():
        pytest.skip("no gfx950 device")
    lib = ctypes.CDLL(os.path.join(REPO, "dip-fmm_amd", "libhipfmm.so"))
    lib.hipfmm_debug_inject_error.argtypes = [ctypes.c_int, ctypes.c_int]
    n = 100000
    x = np.random.default_rng(K).uniform(size=(n, 3))
    o = hip.UniformFmmOptions()
    o.expansion_order, o.tree.max_level = 6, 4
    o.backend = hip.ExecutionBackend.HIP_FULL
    o.precision = hip.StaticPrecision.FLOAT64 if bits == 64 else hip.StaticPrecision.FLOAT32
    o.hip_m2l_mode = getattr(hip.HipM2LMode, mode)
    o.fixed_target_source_indices = range(n)
    f = hip.UniformFmm(x, x, o)
    dtype = torch.float64 if bits == 64 else torch.float32
    bad, good = (torch.randn((K, n, 3), dtype=dtype, device="cuda") for _ in range(2))
    want, out, lost = torch.empty_like(good), torch.empty_like(good), torch.empty_like(good)
    f.evaluate_device(good.data_ptr(), want.data_ptr(), K, torch.cuda.current_stream().cuda_stream)
    host = f.evaluate_batch(good.cpu().numpy().astype(np.float64))
    torch.cuda.synchronize()
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    group = hip.HipGroup([f], [good.data_ptr()], [out.data_ptr()], [K])
    out.fill_(float("nan"))
    torch.cuda.synchronize()
    failures = 0
    for skip in range(200):
        lib.hipfmm_debug_inject_error(HIP_ERROR_LAUNCH_FAILURE, skip)
        try:
            f.evaluate_device(bad.data_ptr(), lost.data_ptr(), K, first.cuda_stream)
            raised = False
        except RuntimeError as e:
            raised = True
            assert "launch failure" in str(e).lower(), str(e)
        finally:
            lib.hipfmm_debug_inject_error(0, 0)
        if not raised:
            break
        failures += 1
        # Straight on: the failed evaluate's kernels would still be running.
        if skip % 3 == 0:
            f.evaluate_device(good.data_ptr(), out.data_ptr(), K, second.cuda_stream)
        elif skip % 3 == 1:
            group.launch(second.cuda_stream)
        else:
            np.testing.assert_array_equal(f.evaluate_batch(good.cpu().numpy().astype(np.float64)), host)
            continue
        torch.cuda.synchronize()
        assert torch.equal(out, want), f"call {skip}"
        out.fill_(float("nan"))
        torch.cuda.synchronize()
    assert failures >= 20  # every checked call of the evaluate in turn
