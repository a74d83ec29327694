"""Evaluates of one plan run in the order of their calls, whatever streams and
entry points they use: each result equals the plan's own one-at-a-time result
bit for bit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 32])
def test_one_plan_on_alternating_streams(K):
    import cdfmm_hip as hip
    import torch

    if not hip.hip_full_available():
        pytest.skip("no gfx950 device")
    n = 20000
    rng = np.random.default_rng(K)
    x = rng.uniform(size=(n, 3))
    o = hip.UniformFmmOptions()
    o.expansion_order, o.tree.max_level = 4, 3
    o.backend, o.precision = hip.ExecutionBackend.HIP_FULL, hip.StaticPrecision.FLOAT32
    o.fixed_target_source_indices = range(n)
    f = hip.UniformFmm(x, x, o)
    moments = [torch.tensor(rng.normal(size=(K, n, 3)), dtype=torch.float32, device="cuda") for _ in range(6)]
    alone = []
    for m in moments:
        out = torch.empty_like(m)
        f.evaluate_device(m.data_ptr(), out.data_ptr(), K, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        alone.append(out)
    host = f.evaluate_batch(moments[0].cpu().numpy().astype(np.float64))
    outs = [torch.full_like(m, float("nan")) for m in moments]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.current_stream(), torch.cuda.Stream()]
    group = hip.HipGroup([f], [moments[5].data_ptr()], [outs[5].data_ptr()], [K])
    for i in range(5):
        f.evaluate_device(moments[i].data_ptr(), outs[i].data_ptr(), K, streams[i % 3].cuda_stream)
    group.launch(streams[0].cuda_stream)
    after = f.evaluate_batch(moments[0].cpu().numpy().astype(np.float64))
    torch.cuda.synchronize()
    for a, b in zip(alone, outs):
        assert torch.equal(a, b)
    np.testing.assert_array_equal(host, after)
