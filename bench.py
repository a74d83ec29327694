#!/usr/bin/env python3
"""HipFull headline benchmark (one MI355X).

Metric: field evaluations per second at 2^20 dipoles, p = 8, K = 32 moment
states -- the MFMA-batched evaluate, reported with the plain-HIP FP32 rate
beside it and the accuracy of the MFMA result.

A step is one batched evaluate of K = 32 moment states on the fixed plan
(2^20 dipoles uniform in [0,1)^3, targets = sources with the identity map,
expansion order 8, uniform depth 5, FP32 plan, M2L on the matrix cores with
bf16 hi/lo split operands).  Moments and fields stay in HBM (torch tensors);
value = N * K * steps / elapsed seconds, the elapsed time between
synchronisations around the timed steps (the same region timed with HIP
events on the caller's stream is reported beside it).  The plain path (M2L
in FP32, on the full-precision matrix instructions, one moment state per
evaluate) is timed on the same plan; speedup_vs_plain is the batched bf16
rate over its rate, so it falls as the plain path gets faster.

Accuracy: rel. L2 of the MFMA result (states 0 and K-1) against the FP64 FMM
at the same (p, depth) (the HipFull FP64 plan, itself checked against
CpuStatic to 1e-12 by the tests) and against the FP64 direct sum on 4096
seeded sample targets.

Roofline: the dominant kernel is the M2L product (one launch over levels
2..5); its algorithmic work is 2 nc^2 flops per list-2 interaction and moment
state, nc = 81 at p = 8 (the class matrices factor through the (p+1)^2-
dimensional harmonic subspace; the reference's form uses n = 165 and is
reported beside it), timed with HIP events on the evaluate's stream around
that launch.

The other benchmark configurations (C2 plain, C3 precision, C4 batching, C5
differentiation; dip-fmm_amd/workloads.py) each get a line under "configs":
their rate and their error against the FP64 FMM and the FP64 direct sum.

CPU baseline: the reference's method (1 warm-up evaluate, then the median of
5 samples of 10 evaluates with distinct seeded states) in a child process
with OMP_PROC_BIND=close, OMP_PLACES=cores: the repository's CpuStatic
restatement (oracle/, "port") on a bounded sample of the headline workload,
the compiled reference itself (oracle/_ref) at C1 when it is present, and
the restatement on a sample of C2.
"""

from __future__ import annotations

import argparse
import json
import os
import subprocess
import sys
import time

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "dip-fmm_amd"))

import workloads as W  # noqa: E402

MFMA_BF16_PEAK_TFLOPS = 2500.0  # MI355X dense BF16 MFMA
SEED = W.seed(2)                # the headline uses C2's geometry and generator


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def make_plan(hip, src, order, depth, precision, mode, tgt=None, ids=True, root=None):
    o = hip.UniformFmmOptions()
    o.expansion_order = order
    o.tree.max_level = depth
    o.backend = hip.ExecutionBackend.HIP_FULL
    o.precision = precision
    if ids:
        o.fixed_target_source_indices = list(range(len(src)))
    o.hip_m2l_mode = mode
    if root is not None:
        o.tree.root_centre = hip.Vec3(*root[:3])
        o.tree.root_half_width = root[3]
    return hip.UniformFmm(src, src if tgt is None else tgt, o)


def rel_l2(a, b) -> float:
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def measured_traffic(n: int, order: int, depth: int, k: int):
    """HBM bytes per M2L launch at the headline workload, from the committed
    rocprofv3 PMC summary (FETCH_SIZE and WRITE_SIZE scaled by a 256 MiB copy);
    None for any other workload."""
    path = os.path.join(HERE, "profiles", "m2l_mfma_1M_p8_d5_K32_traffic.json")
    if (n, order, depth, k) != (1 << 20, 8, 5, 32) or not os.path.exists(path):
        return None
    with open(path) as fh:
        return float(json.load(fh)["traffic_bytes_per_launch"])


# --------------------------------------------------------------------------
# CPU baseline (runs in a child process so that the OpenMP binding applies
# from the start of the runtime).

def _lscpu() -> dict:
    info = {}
    try:
        out = subprocess.run(["lscpu"], capture_output=True, text=True, timeout=20).stdout
        for line in out.splitlines():
            k, _, v = line.partition(":")
            info[k.strip()] = v.strip()
    except (OSError, subprocess.SubprocessError):
        pass
    model = info.get("Model name", "unknown")
    try:
        physical = int(info["Core(s) per socket"]) * int(info["Socket(s)"])
    except (KeyError, ValueError):
        physical = None
    return {"cpu_model": model, "host_physical_cores": physical}


def _cpu_sample(oracle, kind, x, order, depth, precision, output, states) -> dict:
    n = len(x)
    t0 = time.perf_counter()
    f = oracle.CpuFmm(x, x, order, depth, precision, fixed_ids=np.arange(n), kind=kind)
    setup = time.perf_counter() - t0
    f.evaluate(states(0), output=output)  # warm-up
    samples = []
    for s in range(5):
        ms = [states(1 + 10 * s + e) for e in range(10)]
        t0 = time.perf_counter()
        for m in ms:
            f.evaluate(m, output=output)
        samples.append((time.perf_counter() - t0) / 10)
    med = float(np.median(samples))
    return {"setup_s": setup, "median_ms_per_evaluate": 1e3 * med, "samples_ms": [1e3 * s for s in samples],
            "value": n / med}


def cpu_baseline_child() -> dict:
    sys.path.insert(0, os.path.join(HERE, "oracle"))
    import oracle

    threads = int(os.environ.get("OMP_NUM_THREADS", "0")) or len(os.sched_getaffinity(0))
    method = "1 warm-up evaluate, then the median of 5 samples x 10 evaluates, distinct seeded states " \
             "(benchmarks/benchmark_uniform_fmm.cpp:806-831)"
    env = {k: os.environ.get(k) for k in ("OMP_NUM_THREADS", "OMP_PROC_BIND", "OMP_PLACES")}
    # Headline sample: 2^14 dipoles at the headline's density (32 per leaf,
    # depth 3), p = 8, FP32, one state per evaluate.
    n, depth, order = 1 << 14, 3, 8
    x = W.uniform_cube(n, SEED)
    head = _cpu_sample(oracle, "oracle", x, order, depth, 32, "field",
                       lambda k: np.random.default_rng(SEED + 1000 + k).standard_normal((n, 3)))
    log(f"cpu baseline (port, headline sample): {head['median_ms_per_evaluate']:.1f} ms per evaluate")
    out = {
        "value": head["value"],
        "unit": "field evals/s",
        "cores": threads,
        "kind": "port",
        "sample": f"CpuStatic restatement (oracle/), FP32, 2^14 uniform dipoles at the headline's density "
                  f"(32 per leaf, depth 3), p=8, one state per evaluate; {method}",
        "median_ms_per_evaluate": head["median_ms_per_evaluate"],
        "samples_ms": head["samples_ms"],
        "setup_s": head["setup_s"],
        "omp": env,
        **_lscpu(),
    }
    # C1 with the compiled reference (its own sources, oracle/_ref), FP64,
    # field and potential.
    kind = "ref" if oracle.ref_available() else "oracle"
    x1 = W.uniform_cube(20000, W.seed(1))
    c1 = _cpu_sample(oracle, kind, x1, 4, 4, 64, "both",
                     lambda k: W.unit_states(20000, 1, W.seed(1) + 10 * k)[0])
    c1.update({"kind": "reference" if kind == "ref" else "port", "unit": "field+potential evals/s",
               "workload": "C1: 20,000 uniform dipoles, unit moments, p=4, depth 4, FP64, field and potential"})
    out["c1"] = c1
    log(f"cpu baseline C1 ({c1['kind']}): {c1['median_ms_per_evaluate']:.1f} ms per evaluate")
    # C2 sample: 2^14 dipoles at C2's density (32 per leaf, depth 3), p = 6, FP32.
    n2 = 1 << 14
    x2 = W.uniform_cube(n2, W.seed(2))
    c2 = _cpu_sample(oracle, "oracle", x2, 6, 3, 32, "field",
                     lambda k: np.random.default_rng(W.seed(2) + 1000 + k).standard_normal((n2, 3)))
    c2.update({"kind": "port", "unit": "field evals/s",
               "workload": "C2 sample: 2^14 uniform dipoles (32 per leaf, depth 3), p=6, FP32, field"})
    out["c2_sample"] = c2
    log(f"cpu baseline C2 sample (port): {c2['median_ms_per_evaluate']:.1f} ms per evaluate")
    return out


def cpu_baseline() -> dict:
    env = dict(os.environ)
    env.setdefault("OMP_PROC_BIND", "close")
    env.setdefault("OMP_PLACES", "cores")
    proc = subprocess.run([sys.executable, os.path.abspath(__file__), "--cpu-baseline-child"], env=env,
                          capture_output=True, text=True, timeout=900)
    sys.stderr.write(proc.stderr)
    if proc.returncode != 0:
        raise RuntimeError(f"CPU baseline child failed ({proc.returncode})")
    return json.loads(proc.stdout.strip().splitlines()[-1])


# --------------------------------------------------------------------------
# GPU helpers

def time_device(torch, run, reps):
    """Seconds per call of `run` over `reps` calls after one untimed call,
    from HIP events on the caller's stream (every call is ordered on it)."""
    run()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        run()
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) * 1e-3 / reps


def direct_error(hip, x_src, x_tgt, moments, fields, ids, seed):
    """rel. L2 of `fields` against the FP64 direct sum on 4096 seeded targets."""
    sample = W.sample_targets(len(x_tgt), 4096, seed)
    direct = hip.direct_field(x_tgt[sample], x_src, moments, None if ids is None else ids[sample])
    return rel_l2(np.asarray(fields)[sample], direct), sample, direct


def config_c2(hip, torch, stream) -> dict:
    # 2^20 uniform dipoles, p = 6, depth 5, FP32, plain path: 100 seeded
    # states evaluated one by one on the fixed plan.
    n, p, depth, reps = 1 << 20, 6, 5, 100
    x = W.uniform_cube(n, W.seed(2))
    f = make_plan(hip, x, p, depth, hip.StaticPrecision.FLOAT32, hip.HipM2LMode.VALU)
    ms = torch.empty((reps, n, 3), dtype=torch.float32, device="cuda")
    for k in range(reps):
        ms[k] = torch.from_numpy(np.random.default_rng(W.seed(2) + 1000 + k).standard_normal((n, 3),
                                                                                           dtype=np.float32))
    out = torch.empty((reps, n, 3), dtype=torch.float32, device="cuda")
    f.evaluate_device(ms[0].data_ptr(), out[0].data_ptr(), 1, stream)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for k in range(reps):
        f.evaluate_device(ms[k].data_ptr(), out[k].data_ptr(), 1, stream)
    torch.cuda.synchronize()
    sec = (time.perf_counter() - t0) / reps
    h0, h99 = out[0].cpu().numpy(), out[reps - 1].cpu().numpy()
    m0, m99 = ms[0].double().cpu().numpy(), ms[reps - 1].double().cpu().numpy()
    del f, ms, out
    torch.cuda.empty_cache()
    f64 = make_plan(hip, x, p, depth, hip.StaticPrecision.FLOAT64, hip.HipM2LMode.VALU)
    r0 = f64.evaluate(m0)["H"]
    r99 = f64.evaluate(m99)["H"]
    del f64
    e_direct, sample, direct = direct_error(hip, x, x, m0, h0, np.arange(n), W.seed(2))
    res = {
        "workload": "C2: 2^20 uniform dipoles, targets = sources, p=6, depth 5, FP32, plain HIP path (FP32 "
                    "M2L), 1 state per evaluate, 100 seeded states on a fixed plan, device operands",
        "value": n / sec, "unit": "field evals/s", "ms_per_evaluate": 1e3 * sec, "evaluates": reps,
        "accuracy": {"vs_fp64_fmm_state0": rel_l2(h0, r0), "vs_fp64_fmm_state99": rel_l2(h99, r99),
                     "vs_fp64_direct_4096": e_direct, "fp64_fmm_vs_fp64_direct_4096": rel_l2(r0[sample], direct)},
    }
    log(f"C2: {res['ms_per_evaluate']:.2f} ms per evaluate, {res['value']:.3e} evals/s, {res['accuracy']}")
    return res


def config_c3(hip, torch, stream) -> dict:
    # 2^20 dipoles, 80% in 64 Gaussian blobs, p = 8, depth 6: the four M2L
    # arithmetics (FP64 plan; FP32 plan with full FP32, bf16 hi/lo and
    # fp16 level-scaled hi/lo on the matrix cores) against the FP64 direct
    # sum on 4096 seeded targets.  The matrix-core modes run K = 32 states.
    n, p, depth, K = 1 << 20, 8, 6, 32
    x = W.gaussian_blobs(n, W.seed(3))
    ids = np.arange(n)
    ms = torch.from_numpy(W.normal_states(n, K, W.seed(3), dtype=np.float32)).cuda()
    f = make_plan(hip, x, p, depth, hip.StaticPrecision.FLOAT32, hip.HipM2LMode.MFMA_BF16X3)
    out = torch.empty((K, n, 3), dtype=torch.float32, device="cuda")
    modes = {}
    for name, mode, k in (("bf16x3", hip.HipM2LMode.MFMA_BF16X3, K), ("fp16x3", hip.HipM2LMode.MFMA_FP16X3, K),
                          ("fp32_valu", hip.HipM2LMode.VALU, 1)):
        f.set_m2l_mode(mode)
        sec = time_device(torch, lambda: f.evaluate_device(ms.data_ptr(), out.data_ptr(), k, stream), 3)
        modes[name] = {"batch": k, "ms_per_evaluate": 1e3 * sec, "value": n * k / sec,
                       "fields": out[0].cpu().numpy().copy()}
    m0 = ms[0].double().cpu().numpy()
    del f, ms, out
    torch.cuda.empty_cache()
    f64 = make_plan(hip, x, p, depth, hip.StaticPrecision.FLOAT64, hip.HipM2LMode.VALU)
    t0 = time.perf_counter()
    r0 = f64.evaluate(m0)["H"]
    sec64 = time.perf_counter() - t0
    del f64
    e64, sample, direct = direct_error(hip, x, x, m0, r0, ids, W.seed(3))
    modes["fp64"] = {"batch": 1, "ms_per_evaluate": 1e3 * sec64, "value": n / sec64,
                     "note": "host operands, transfers included"}
    for name, v in modes.items():
        h = v.pop("fields", None)
        v["vs_fp64_direct_4096"] = e64 if h is None else rel_l2(h[sample], direct)
        if h is not None:
            v["vs_fp64_fmm"] = rel_l2(h, r0)
    res = {"workload": "C3: 2^20 dipoles, 80% in 64 Gaussian blobs (sigma 0.02) + 20% uniform, p=8, depth 6, "
                       "M2L in FP64 / FP32 / bf16 hi-lo / fp16 level-scaled, error vs FP64 direct on 4096 targets",
           "modes": modes}
    log("C3: " + ", ".join(f"{k} {v['ms_per_evaluate']:.1f} ms (K={v['batch']}) direct {v['vs_fp64_direct_4096']:.2e}"
                           for k, v in modes.items()))
    return res


def config_c4(hip, torch, stream) -> dict:
    # 128^3 jittered lattice, wave moment states, p = 6, FP32 with the bf16
    # matrix-core M2L, K in {1, 8, 32, 64}, depths 5 and 6; and 8 uniform
    # cubes of N log-uniform in [16k, 1M] in one group launch.
    side, p = 128, 6
    x = W.jittered_lattice(side, W.seed(4))
    n = len(x)
    ids = np.arange(n)
    ms = torch.from_numpy(W.wave_states(x, 64, W.seed(4), dtype=np.float32)).cuda()
    out = torch.empty((64, n, 3), dtype=torch.float32, device="cuda")
    res = {"workload": "C4: 128^3 jittered lattice (2,097,152 dipoles), wave moment states, p=6, FP32, bf16 hi/lo "
                       "M2L on the matrix cores; 8 uniform cubes of N log-uniform in [16k, 1M] in one group launch"}
    for depth in (5, 6):
        f = make_plan(hip, x, p, depth, hip.StaticPrecision.FLOAT32, hip.HipM2LMode.MFMA_BF16X3)
        rates = {}
        for K in (1, 8, 32, 64):
            sec = time_device(torch, lambda: f.evaluate_device(ms.data_ptr(), out.data_ptr(), K, stream), 3)
            rates[f"K{K}"] = {"ms_per_evaluate": 1e3 * sec, "value": n * K / sec}
        h0 = out[0].cpu().numpy()
        del f
        torch.cuda.empty_cache()
        m0 = ms[0].double().cpu().numpy()
        f64 = make_plan(hip, x, p, depth, hip.StaticPrecision.FLOAT64, hip.HipM2LMode.VALU)
        r0 = f64.evaluate(m0)["H"]
        del f64
        e, sample, direct = direct_error(hip, x, x, m0, h0, ids, W.seed(4))
        res[f"depth{depth}"] = {"rates": rates, "accuracy": {
            "vs_fp64_fmm_state0": rel_l2(h0, r0), "vs_fp64_direct_4096": e,
            "fp64_fmm_vs_fp64_direct_4096": rel_l2(r0[sample], direct)}}
        log(f"C4 depth {depth}: " + ", ".join(f"{k} {v['value']:.3e}" for k, v in rates.items()) +
            f"; {res[f'depth{depth}']['accuracy']}")
    del ms, out
    torch.cuda.empty_cache()
    sizes = W.log_uniform_sizes(8, 16384, 1 << 20, W.seed(4))
    fmms, moms, outs = [], [], []
    for i, ng in enumerate(sizes):
        xg = W.uniform_cube(int(ng), W.seed(4) + 100 + i)
        depth = int(np.clip(np.round(np.log(ng / 32) / np.log(8)), 2, 5))
        fmms.append(make_plan(hip, xg, p, depth, hip.StaticPrecision.FLOAT32, hip.HipM2LMode.MFMA_BF16X3))
        moms.append(torch.from_numpy(W.normal_states(int(ng), 32, W.seed(4) + 100 + i, dtype=np.float32)).cuda())
        outs.append(torch.empty((32, int(ng), 3), dtype=torch.float32, device="cuda"))
    group = hip.HipGroup(fmms, [m.data_ptr() for m in moms], [o.data_ptr() for o in outs], [32] * 8)

    def sequential():
        for f, m, o in zip(fmms, moms, outs):
            f.evaluate_device(m.data_ptr(), o.data_ptr(), 32, stream)

    s_seq = time_device(torch, sequential, 3)
    s_grp = time_device(torch, lambda: group.launch(stream), 3)
    evals = 32 * int(sizes.sum())
    res["group_of_8"] = {"sizes": [int(v) for v in sizes], "batch": 32, "ms_group": 1e3 * s_grp,
                         "ms_sequential": 1e3 * s_seq, "value": evals / s_grp}
    log(f"C4 group of 8: {1e3 * s_grp:.2f} ms against {1e3 * s_seq:.2f} ms one after another")
    del group, fmms, moms, outs
    torch.cuda.empty_cache()
    return res


def config_c5(hip, torch, stream) -> dict:
    # 262,144 slab sources, 65,536 plane targets, p = 6, depth 5, FP32 (bf16
    # matrix-core M2L): the gradient of L = 0.5 |H(m) - H_target|^2 with
    # respect to the moments (adjoint pass) and the target positions (field
    # gradient), one state.  Central differences are in the GPU tests.
    import cdfmm_hip

    ns, side, p, depth = 262144, 256, 6, 5
    src = W.slab_sources(ns, W.seed(5))
    tgt = W.plane_targets(side, W.seed(5))
    nt = len(tgt)
    root = (0.5, 0.5, 0.1, 0.5)
    states = W.normal_states(ns, 2, W.seed(5))
    f = make_plan(hip, src, p, depth, hip.StaticPrecision.FLOAT32, hip.HipM2LMode.MFMA_BF16X3, tgt=tgt, ids=False,
                  root=root)
    m_t = torch.tensor(states[0], dtype=torch.float32, device="cuda")
    h_target = cdfmm_hip.dipole_field(f, m_t).detach()
    m = torch.tensor(states[1], dtype=torch.float32, device="cuda")

    def gradient():
        mv = m.clone().requires_grad_(True)
        h = cdfmm_hip.dipole_field(f, mv)
        loss = 0.5 * ((h - h_target) ** 2).sum()
        loss.backward()
        d_t, _ = cdfmm_hip.position_gradients(f, m[None], (h.detach() - h_target)[None])
        return mv.grad, d_t

    sec_fwd = time_device(torch, lambda: cdfmm_hip.dipole_field(f, m), 5)
    sec_grad = time_device(torch, gradient, 5)
    h = cdfmm_hip.dipole_field(f, m).cpu().numpy()
    e, _, _ = direct_error(hip, src, tgt, states[1], h, None, W.seed(5))
    res = {"workload": "C5: 262,144 sources in the slab [0,1]^2 x [0,0.1], 65,536 targets on a jittered 256^2 grid "
                       "at z=0.2, p=6, depth 5, FP32 (bf16 hi/lo M2L); loss 0.5|H(m)-H_target|^2, dL/dm and "
                       "dL/d(target positions)",
           "forward_ms": 1e3 * sec_fwd, "loss_and_gradients_ms": 1e3 * sec_grad,
           "value": nt / sec_grad, "unit": "target gradients/s (loss, dL/dm and dL/dx_t per target)",
           "accuracy": {"field_vs_fp64_direct_4096": e}}
    log(f"C5: forward {1e3 * sec_fwd:.2f} ms, loss + gradients {1e3 * sec_grad:.2f} ms, field vs direct {e:.2e}")
    return res


def main() -> int:
    ap = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--n", type=int, default=1 << 20)
    ap.add_argument("--order", type=int, default=8)
    ap.add_argument("--depth", type=int, default=5)
    ap.add_argument("--batch", type=int, default=32)
    ap.add_argument("--plain-steps", type=int, default=3)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-accuracy", action="store_true")
    ap.add_argument("--no-plain", action="store_true")
    ap.add_argument("--no-fp16", action="store_true", help="skip the FP16-split M2L line")
    ap.add_argument("--autotune", action="store_true",
                    help="run the plan's launch autotuner at K states before timing")
    ap.add_argument("--near-variant", type=int, default=0,
                    help="pin the near-field kernel (codes of hip_plan_statistics; 0 = built-in default)")
    ap.add_argument("--no-other-paths", action="store_true",
                    help="skip the adjoint, potential and field-gradient timings")
    ap.add_argument("--configs", default="c2,c3,c4,c5",
                    help="comma-separated benchmark configurations to report beside the headline ('' for none)")
    ap.add_argument("--copy-calibration-mib", type=int, default=0,
                    help="run one device-to-device copy of this many MiB before the steps (the reference kernel "
                         "for scaling PMC byte counters)")
    ap.add_argument("--cpu-baseline-child", action="store_true", help=argparse.SUPPRESS)
    args = ap.parse_args()

    if args.cpu_baseline_child:
        print(json.dumps(cpu_baseline_child()), flush=True)
        return 0

    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print("bench.py measures one GPU: the HipFull evaluate runs on a single MI355X and the library has no "
              "multi-GPU path; run with --gpus 1.", file=sys.stderr)
        return 2

    import torch
    import cdfmm_hip as hip

    if not hip.hip_full_available():
        raise RuntimeError("HipFull needs a gfx950 device")
    dev = torch.device("cuda:0")
    N, K, p, depth = args.n, args.batch, args.order, args.depth
    log(f"device: {hip.hip_device_description()}")
    t0 = time.perf_counter()
    x = W.uniform_cube(N, SEED)
    fmm = make_plan(hip, x, p, depth, hip.StaticPrecision.FLOAT32, hip.HipM2LMode.MFMA_BF16X3)
    if args.near_variant:
        fmm.set_launch_choices(0, args.near_variant)
    if args.autotune:
        fmm.autotune(K)
        st = fmm.hip_plan_statistics
        log(f"autotune: M2L tile shape {st['m2l_tile_shape']}, near-field variant {st['p2p_kernel_variant']} "
            f"in {st['autotune_seconds']:.1f}s")
    log(f"plan setup: {time.perf_counter() - t0:.1f}s")
    stats = fmm.hip_plan_statistics
    moments = torch.from_numpy(W.normal_states(N, K, SEED, dtype=np.float32)).to(dev)
    fields = torch.empty((K, N, 3), dtype=torch.float32, device=dev)
    stream = torch.cuda.current_stream().cuda_stream

    def step():
        fmm.evaluate_device(moments.data_ptr(), fields.data_ptr(), K, stream)

    if args.copy_calibration_mib > 0:
        src = torch.ones(args.copy_calibration_mib << 18, dtype=torch.float32, device=dev)
        dst = torch.empty_like(src)
        dst.copy_(src)
        torch.cuda.synchronize()
        log(f"copy calibration: {args.copy_calibration_mib} MiB read + {args.copy_calibration_mib} MiB written")
        del src, dst

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    # Every M2L launch is timed by its own pair of HIP events on the plan's
    # stream; the difference of the running totals around the timed region
    # gives that region's average launch time without synchronising steps.
    before = fmm.device_timings()
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t_start = time.perf_counter()
    ev0.record()
    for _ in range(args.steps):
        step()
    ev1.record()
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t_start
    ms_per_step = 1e3 * elapsed / args.steps
    ms_per_step_events = ev0.elapsed_time(ev1) / args.steps
    value = N * K * args.steps / elapsed
    stage = fmm.device_timings()
    launches = stage["m2l_kernel_launches"] - before["m2l_kernel_launches"]
    if launches != args.steps:
        raise RuntimeError(f"expected {args.steps} M2L launches in the timed region, saw {launches}")
    m2l_s = (stage["m2l_kernel_total"] - before["m2l_kernel_total"]) / launches
    log(f"MFMA K={K}: {ms_per_step:.2f} ms/step ({ms_per_step_events:.2f} ms by events), {value:.3e} evals/s; "
        f"stages {stage}")

    pairs = stats["m2l_interaction_count"]
    n = fmm.coefficient_count
    nc = int(stats["m2l_operand_size"])  # (p+1)^2 when the class matrices factor through the harmonic subspace
    m2l_flops = 2.0 * nc * nc * pairs * K
    achieved = m2l_flops / m2l_s / 1e12
    roofline = {
        "bound": "mfma",
        "achieved": achieved,
        "peak": MFMA_BF16_PEAK_TFLOPS,
        "unit": "TFLOP/s",
        "frac": achieved / MFMA_BF16_PEAK_TFLOPS,
        "traffic": measured_traffic(N, p, depth, K),
        "kernel": "m2l_mfma_kernel (one launch, levels 2..L, the last level's inner class dispatched first)",
        "kernel_ms": 1e3 * m2l_s,
        "algorithmic_flops_per_launch": m2l_flops,
        "m2l_operand_size": nc,
        "reference_equivalent_flops_per_launch": 2.0 * n * n * pairs * K,
        "list2_interactions": pairs,
        "split_products_per_flop": 3,
    }

    checked = (0, K - 1)
    result_fields = {k: fields[k].float().cpu().numpy() for k in checked}
    plain = {}
    if not args.no_plain:
        fmm.set_m2l_mode(hip.HipM2LMode.VALU)
        one_m = moments[0:1].contiguous()
        one_f = torch.empty((1, N, 3), dtype=torch.float32, device=dev)
        fmm.evaluate_device(one_m.data_ptr(), one_f.data_ptr(), 1, stream)
        torch.cuda.synchronize()
        tp = time.perf_counter()
        for _ in range(args.plain_steps):
            fmm.evaluate_device(one_m.data_ptr(), one_f.data_ptr(), 1, stream)
        torch.cuda.synchronize()
        plain_s = (time.perf_counter() - tp) / args.plain_steps
        pt = fmm.device_timings()
        plain = {"value": N / plain_s, "ms_per_evaluate": 1e3 * plain_s, "m2l_kernel_ms": 1e3 * pt["m2l_kernel"]}
        plain_fields = one_f[0].cpu().numpy()
        # The plain path at the headline's batch: the same K = 32 states in
        # one evaluate with the FP32 M2L.
        s32 = time_device(torch, step, max(1, min(args.plain_steps, 3)))
        plain["k32"] = {"value": N * K / s32, "ms_per_step": 1e3 * s32,
                        "m2l_kernel_ms": 1e3 * fmm.device_timings()["m2l_kernel"]}
        fmm.set_m2l_mode(hip.HipM2LMode.MFMA_BF16X3)
        log(f"plain FP32 K=1: {1e3 * plain_s:.2f} ms/evaluate, {N / plain_s:.3e} evals/s; "
            f"K={K}: {1e3 * s32:.2f} ms/step")

    # The same step with the level-scaled FP16 hi/lo M2L (same MFMA rate,
    # 22 bits per operand instead of 16), reported beside the headline.
    fp16 = {}
    fp16_fields = None
    if not args.no_fp16:
        fmm.set_m2l_mode(hip.HipM2LMode.MFMA_FP16X3)
        s16 = time_device(torch, step, max(1, min(args.steps, 5)))
        fp16 = {"value": N * K / s16, "ms_per_step": 1e3 * s16}
        fp16_fields = fields[0].float().cpu().numpy()
        fmm.set_m2l_mode(hip.HipM2LMode.MFMA_BF16X3)
        log(f"MFMA FP16x3 K={K}: {1e3 * s16:.2f} ms/step, {N * K / s16:.3e} evals/s")

    # The other device paths of the same plan at the same workload: the
    # adjoint (cotangents in, moment gradients out), fields with potentials,
    # and the field gradient (6 entries per target).
    other = {}
    if not args.no_other_paths:
        reps = max(1, min(args.steps, 3))
        grad = torch.empty_like(moments)
        sec = time_device(torch, lambda: fmm.evaluate_adjoint_device(fields.data_ptr(), grad.data_ptr(), K, stream),
                          reps)
        other["adjoint"] = {"ms_per_step": 1e3 * sec, "value": N * K / sec}
        del grad
        pot = torch.empty((K, N), dtype=torch.float32, device=dev)
        sec = time_device(torch, lambda: fmm.evaluate_potential_device(moments.data_ptr(), fields.data_ptr(),
                                                                       pot.data_ptr(), K, stream), reps)
        other["fields_and_potentials"] = {"ms_per_step": 1e3 * sec, "value": N * K / sec}
        del pot
        gmat = torch.empty((K, N, 6), dtype=torch.float32, device=dev)
        sec = time_device(torch, lambda: fmm.evaluate_field_gradient_device(moments.data_ptr(), gmat.data_ptr(), K,
                                                                            stream), reps)
        other["field_gradient"] = {"ms_per_step": 1e3 * sec, "value": N * K / sec}
        del gmat
        torch.cuda.empty_cache()
        log("other paths (ms per K-state step): " + ", ".join(f"{k} {v['ms_per_step']:.2f}" for k, v in other.items()))

    accuracy = {}
    if not args.no_accuracy:
        m_checked = {k: moments[k].double().cpu().numpy() for k in checked}
        del fmm, moments, fields
        torch.cuda.empty_cache()
        f64 = make_plan(hip, x, p, depth, hip.StaticPrecision.FLOAT64, hip.HipM2LMode.VALU)
        ref64 = {k: f64.evaluate(m_checked[k])["H"] for k in checked}
        del f64
        accuracy["mfma_vs_fp64_fmm"] = rel_l2(result_fields[0], ref64[0])
        accuracy[f"mfma_vs_fp64_fmm_state{K - 1}"] = rel_l2(result_fields[K - 1], ref64[K - 1])
        if plain:
            accuracy["plain_fp32_vs_fp64_fmm"] = rel_l2(plain_fields, ref64[0])
        if fp16_fields is not None:
            accuracy["mfma_fp16x3_vs_fp64_fmm"] = rel_l2(fp16_fields, ref64[0])
        e, sample, direct = direct_error(hip, x, x, m_checked[0], result_fields[0], np.arange(N), SEED)
        accuracy["mfma_vs_fp64_direct_4096"] = e
        accuracy["fp64_fmm_vs_fp64_direct_4096"] = rel_l2(ref64[0][sample], direct)
        log(f"accuracy: {accuracy}")
    else:
        del fmm, moments, fields
    torch.cuda.empty_cache()

    configs = {}
    for name in [c for c in args.configs.split(",") if c]:
        run = {"c2": config_c2, "c3": config_c3, "c4": config_c4, "c5": config_c5}.get(name)
        if run is None:
            raise SystemExit(f"unknown configuration {name!r}")
        t0 = time.perf_counter()
        configs[name] = run(hip, torch, stream)
        configs[name]["bench_seconds"] = time.perf_counter() - t0
        torch.cuda.empty_cache()

    baseline = None if args.no_cpu_baseline else cpu_baseline()

    line = {
        "metric": "field evals/s, 1M dipoles p=8 K=32: MFMA-batched vs plain HIP @ rel err≤1e-5",
        "value": value,
        "unit": "field evals/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "ms_per_step_events": ms_per_step_events,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic: uniform [0,1)^3 positions, N(0,1) moment components, seeded",
        "config": {
            "workload": f"{N} dipoles, targets = sources (identity map), p={p}, uniform depth {depth}, "
                        f"K={K} moment states per evaluate, FP32 plan, M2L on MFMA (bf16 hi/lo x3, fp32 accumulate)",
            "n": N, "order": p, "depth": depth, "batch": K, "m2l": "mfma_bf16x3",
        },
        "plain_hip_fp32": plain or None,
        "mfma_fp16x3": fp16 or None,
        "other_paths": other or None,
        "speedup_vs_plain": (value / plain["value"]) if plain else None,
        "accuracy": accuracy or None,
        "stages_ms": {k: 1e3 * v for k, v in stage.items() if k not in ("evaluations", "m2l_kernel_launches")},
        "roofline": roofline,
        "configs": configs or None,
        "cpu_baseline": baseline,
    }
    print(json.dumps(line), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
