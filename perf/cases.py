"""Performance cases of the HipFull evaluate: what a program asks of one plan
(or a group of plans) through the public entry points, from a thousand points
and one moment state to two million points or 64 states.

A case is a dict of plain values:
  entry      field | both | adjoint | gradient (device-resident entry points of
             UniformFmm), host (UniformFmm.evaluate on numpy arrays), loss (the
             torch autograd caller with position gradients), group (HipGroup)
  geometry   uniform | blobs | lattice (targets = sources with the identity
             map) | slab (sources in a slab, targets on a plane above it)
  n, p, depth, k, bits (32 | 64), mode (VALU | MFMA_BF16X3 | MFMA_FP16X3, the
             M2L arithmetic), plans (1; the member count of a group)
"""

import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dip-fmm_amd"))

import cdfmm_hip as hip  # noqa: E402
import workloads as W  # noqa: E402

_DEFAULTS = {"entry": "field", "geometry": "uniform", "bits": 32, "mode": "VALU", "k": 1, "plans": 1}
_SLAB_ROOT = (0.5, 0.5, 0.1, 0.5)  # root box (centre, half-width) that holds the slab and the plane


def _case(**values):
    return {**_DEFAULTS, **values}


def listed():
    return [
        # One moment state on a few points with the default options: a step of
        # a small simulation, where the latency of the whole call counts.
        _case(name="small_1k", n=1000, p=4, depth=2),
        # Fields and potentials in double precision through the drop-in host
        # interface: numpy arrays in and out (20,000 dipoles, p = 4).
        _case(name="host_fp64_20k", entry="host", n=20000, p=4, depth=4, bits=64),
        # A few states on an odd number of points, fields with potentials.
        _case(name="ragged_both_50k", entry="both", n=50021, p=6, depth=4, k=5, mode="MFMA_BF16X3"),
        # The transpose for a batch of cotangents that fills no tile of 32.
        _case(name="adjoint_131k_k20", entry="adjoint", n=131075, p=8, depth=4, k=20, mode="MFMA_FP16X3"),
        # Gradient-based fitting: loss, moment gradient and target position
        # gradient of slab sources seen from a plane.
        _case(name="slab_loss_262k", entry="loss", geometry="slab", n=262144, p=6, depth=5, mode="MFMA_BF16X3"),
        # Field gradients of a batch (forces on dipoles).
        _case(name="gradient_200k_k32", entry="gradient", n=200000, p=6, depth=4, k=32, mode="MFMA_BF16X3"),
        # Double precision on device memory: reference solutions.
        _case(name="fp64_262k", n=262144, p=8, depth=4, bits=64),
        # One state per call on a million points with the default options: an
        # iterative solver or a time step.
        _case(name="plain_1m", n=1 << 20, p=6, depth=5),
        # Uneven geometries in one group launch.
        _case(name="group_of_8", entry="group", n=1 << 18, p=6, depth=4, k=32, mode="MFMA_BF16X3", plans=8),
        # The headline batch: 32 states on a million points at p = 8.
        _case(name="batch_1m_k32", n=1 << 20, p=8, depth=5, k=32, mode="MFMA_BF16X3"),
        # A large lattice with a handful of states.
        _case(name="lattice_2m_k8", geometry="lattice", n=1 << 21, p=6, depth=5, k=8, mode="MFMA_BF16X3"),
        # Clustered points: leaves from empty to hundreds of points.
        _case(name="blobs_1m_k32", geometry="blobs", n=1 << 20, p=8, depth=6, k=32, mode="MFMA_BF16X3"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _depth(n, per_leaf):
    return max(2, min(6, round(math.log(max(n / per_leaf, 1.0)) / math.log(8.0))))


def draw(rng):
    entry = rng.choices(["field", "both", "adjoint", "gradient", "host", "loss", "group"], [8, 3, 3, 2, 2, 2, 1])[0]
    bits = 64 if entry != "loss" and entry != "group" and rng.random() < 0.2 else 32
    k = 1 if entry == "host" or rng.random() < 0.4 else _log_uniform(rng, 2, 64)
    most = 1 << 18 if bits == 64 else 1 << 20
    n = _log_uniform(rng, 1000, most)
    cap = (1 << 20 if bits == 64 else 1 << 24) // (4 if entry in ("gradient", "loss", "group") else 1)
    geometry = "slab" if entry == "loss" else rng.choices(["uniform", "blobs", "lattice", "slab"], [6, 2, 1, 1])[0]
    if geometry == "blobs":
        cap //= 4
    n = max(1000, min(n, cap // k))
    if geometry == "lattice":
        n = round(n ** (1 / 3)) ** 3
    depth = _depth(n, rng.uniform(16, 64)) + (1 if geometry == "blobs" else 0)
    mode = "VALU" if bits == 64 else rng.choice(["VALU", "MFMA_BF16X3", "MFMA_BF16X3", "MFMA_FP16X3"])
    return _case(entry=entry, geometry=geometry, n=n, p=rng.randint(4, 8), depth=min(6, depth), k=k, bits=bits, mode=mode,
                 plans=rng.randint(2, 8) if entry == "group" else 1)


def _member(case, i):
    """Size and depth of member i of a group: uneven sizes up to n."""
    if case["plans"] == 1:
        return case["n"], case["depth"]
    n = max(1000, int(case["n"] * 16.0 ** (-i / (case["plans"] - 1))))
    return n, _depth(n, 40)


def _points(case, n, seed):
    """Sources and targets (the same array where they are the same points)."""
    if case["geometry"] == "slab":
        return W.slab_sources(n, seed), W.plane_targets(max(8, int(math.sqrt(n / 4))), seed)
    if case["geometry"] == "blobs":
        x = W.gaussian_blobs(n, seed)
    elif case["geometry"] == "lattice" and round(n ** (1 / 3)) ** 3 == n:
        x = W.jittered_lattice(round(n ** (1 / 3)), seed)
    else:
        x = W.uniform_cube(n, seed)
    return x, x


def _plan(case, src, tgt, depth):
    o = hip.UniformFmmOptions()
    o.expansion_order = case["p"]
    o.tree.max_level = depth
    o.backend = hip.ExecutionBackend.HIP_FULL
    o.precision = hip.StaticPrecision.FLOAT64 if case["bits"] == 64 else hip.StaticPrecision.FLOAT32
    o.hip_m2l_mode = getattr(hip.HipM2LMode, case["mode"])
    if src is tgt:
        o.fixed_target_source_indices = range(len(src))
    else:
        o.tree.root_centre = hip.Vec3(*_SLAB_ROOT[:3])
        o.tree.root_half_width = _SLAB_ROOT[3]
    return hip.UniformFmm(src, tgt, o)


def _normal(shape, seed, dtype):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(shape, generator=g, dtype=dtype, device="cuda")


def _inputs(case, seed, i=0):
    """Points, and the moments (or cotangents) of member i."""
    n, _ = _member(case, i)
    seed = 100 * seed + i
    src, tgt = _points(case, n, seed)
    rows = len(tgt) if case["entry"] == "adjoint" else len(src)
    dtype = torch.float64 if case["bits"] == 64 else torch.float32
    x = _normal((case["k"], rows, 3), seed + 50, dtype)
    if case["entry"] == "host":  # unit vectors, one state
        x = torch.nn.functional.normalize(x, dim=2)[0].double()
    return src, tgt, x


def prepare(case, seed):
    entry, k = case["entry"], case["k"]
    if entry == "group":
        state = {"entry": entry, "plans": [], "moments": [], "fields": []}
        for i in range(case["plans"]):
            src, tgt, x = _inputs(case, seed, i)
            state["plans"].append(_plan(case, src, tgt, _member(case, i)[1]))
            state["moments"].append(x)
            state["fields"].append(torch.empty((k, len(tgt), 3), dtype=x.dtype, device="cuda"))
        state["group"] = hip.HipGroup(state["plans"], [m.data_ptr() for m in state["moments"]],
                                      [f.data_ptr() for f in state["fields"]], [k] * case["plans"])
        return state
    src, tgt, x = _inputs(case, seed)
    fmm = _plan(case, src, tgt, case["depth"])
    state = {"entry": entry, "fmm": fmm, "x": x, "k": k}
    if entry == "host":
        state["x"] = x.cpu().numpy()
    elif entry == "loss":
        state["measured"] = hip.dipole_field(fmm, _normal(x.shape, 100 * seed + 60, x.dtype)).detach()
    else:
        rows = len(src) if entry == "adjoint" else len(tgt)
        state["out"] = torch.empty((k, rows, 6 if entry == "gradient" else 3), dtype=x.dtype, device="cuda")
        if entry == "both":
            state["phi"] = torch.empty((k, rows), dtype=x.dtype, device="cuda")
    return state


def run(state):
    entry = state["entry"]
    if entry == "group":
        state["group"].launch(torch.cuda.current_stream().cuda_stream)
        return state["fields"]
    fmm, x = state["fmm"], state["x"]
    if entry == "host":
        r = fmm.evaluate(x, output="both")
        return {"H": r["H"], "phi": r["phi"]}
    if entry == "loss":
        m = x.detach().requires_grad_(True)
        h = hip.dipole_field(fmm, m)
        residual = h - state["measured"]
        (0.5 * residual.square().sum()).backward()
        moved, _ = hip.position_gradients(fmm, x, residual.detach())
        return {"moments": m.grad, "targets": moved}
    out, k, stream = state["out"], state["k"], torch.cuda.current_stream().cuda_stream
    if entry == "field":
        fmm.evaluate_device(x.data_ptr(), out.data_ptr(), k, stream)
    elif entry == "adjoint":
        fmm.evaluate_adjoint_device(x.data_ptr(), out.data_ptr(), k, stream)
    elif entry == "gradient":
        fmm.evaluate_field_gradient_device(x.data_ptr(), out.data_ptr(), k, stream)
    else:
        fmm.evaluate_potential_device(x.data_ptr(), out.data_ptr(), state["phi"].data_ptr(), k, stream)
        return {"H": out, "phi": state["phi"]}
    return out


def _leaf_counts(x, depth, lo, width):
    nb = 1 << depth
    c = np.clip(((x - lo) / width * nb).astype(np.int64), 0, nb - 1)
    return np.bincount((c[:, 0] * nb + c[:, 1]) * nb + c[:, 2], minlength=nb ** 3).reshape(nb, nb, nb)


def _neighbourhood(a):
    """Sums over the clipped 3 x 3 x 3 cubes."""
    for axis in range(3):
        pad = [(1, 1) if i == axis else (0, 0) for i in range(3)]
        b = np.pad(a, pad)
        cut = [slice(None)] * 3
        parts = []
        for s in range(3):
            cut[axis] = slice(s, s + a.shape[axis])
            parts.append(b[tuple(cut)])
        a = parts[0] + parts[1] + parts[2]
    return a


def work(case):
    """Inputs read and outputs written once; the near-field products (18 per
    pair and state with the pair tensor formed once) and, per pair of boxes of
    list 2 that hold points, the (p + 1)^2 x (p + 1)^2 product."""
    size, passes = case["bits"] // 8, {"loss": 4}.get(case["entry"], 1)
    moved, flops = 0.0, 0.0
    for i in range(case["plans"]):
        n, depth = _member(case, i)
        src, tgt = _points(case, n, 7)
        lo, width = (np.array(_SLAB_ROOT[:3]) - _SLAB_ROOT[3], 2 * _SLAB_ROOT[3]) if src is not tgt else (0.0, 1.0)
        s, t = _leaf_counts(src, depth, lo, width), _leaf_counts(tgt, depth, lo, width)
        pairs = float((t * _neighbourhood(s)).sum())
        boxes = 0.0
        for level in range(depth, 1, -1):
            full, near = np.sign(s), _neighbourhood(np.sign(s))
            up = full.reshape(full.shape[0] // 2, 2, full.shape[1] // 2, 2, full.shape[2] // 2, 2).sum(axis=(1, 3, 5))
            wide = _neighbourhood(up).repeat(2, 0).repeat(2, 1).repeat(2, 2)
            boxes += float((np.sign(t) * (wide - near)).sum())
            s, t = (a.reshape(a.shape[0] // 2, 2, a.shape[1] // 2, 2, a.shape[2] // 2, 2).sum(axis=(1, 3, 5))
                    for a in (s, t))
        out = {"both": 4, "host": 4, "gradient": 6, "loss": 3}.get(case["entry"], 3)
        moved += case["k"] * (3 * len(src) + out * len(tgt)) * size + 3 * (len(src) + len(tgt)) * size
        if case["entry"] == "loss":
            moved += case["k"] * 3 * (len(src) + len(tgt)) * size
        products = 36 if case["entry"] == "gradient" else 24 if out == 4 else 18
        flops += passes * case["k"] * (products * pairs + 2.0 * (case["p"] + 1) ** 4 * boxes) + 25.0 * passes * pairs
    return {"bytes": moved, "flops": flops}


def _direct(targets, sources, x, same, what):
    """Direct sum in 64 bits of the dipoles x (K, sources, 3): fields (K, N,
    3), with potentials for "both", or field gradients (K, N, 6)."""
    t, s = (torch.as_tensor(a, dtype=torch.float64, device="cuda") for a in (targets, sources))
    m = [x[:, :, c].t().contiguous() for c in range(3)]  # (sources, K)
    k, rows = x.shape[0], {"gradient": 6, "both": 4}.get(what, 3)
    out = torch.zeros((len(t), rows, k), dtype=torch.float64, device="cuda")
    ct, cs = 4096, 16384
    for i in range(0, len(t), ct):
        for j in range(0, len(s), cs):
            r = [t[i:i + ct, None, c] - s[None, j:j + cs, c] for c in range(3)]
            r2 = r[0] * r[0] + r[1] * r[1] + r[2] * r[2]
            lo, hi = max(i, j), min(i + ct, j + cs, len(t))
            if same and lo < hi:
                own = torch.arange(lo, hi, device="cuda")
                r2[own - i, own - j] = math.inf
            f = r2.pow(-1.5) / (4.0 * math.pi)
            mj = [c[j:j + cs] for c in m]
            acc = out[i:i + ct]
            if what == "gradient":
                g = 3.0 * f / r2
                for e, (a, b) in enumerate(((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))):
                    for d in range(3):
                        w = -5.0 * r[a] * r[b] * r[d] / r2
                        for u, v, o in ((a, b, d), (a, d, b), (b, d, a)):
                            if u == v:
                                w = w + r[o]
                        acc[:, e] += (g * w) @ mj[d]
                continue
            for a in range(3):
                fr = f * r[a]
                if what == "both":
                    acc[:, 3] += fr @ mj[a]
                fr = 3.0 * fr / r2
                for b in range(a, 3):
                    w = fr * r[b]
                    if a == b:
                        acc[:, a] += (w - f) @ mj[a]
                    else:
                        acc[:, a] += w @ mj[b]
                        acc[:, b] += w @ mj[a]
    return out.permute(2, 0, 1).contiguous()


def exact(case, seed):
    """The direct sum over all pairs: what the multipole expansion stands for."""
    entry, pairs = case["entry"], 0
    if entry == "group":
        sums = []
        for i in range(case["plans"]):
            pairs += _member(case, i)[0] ** 2
        if pairs > 7e10:
            return None
        for i in range(case["plans"]):
            src, tgt, x = _inputs(case, seed, i)
            sums.append(_direct(tgt, src, x.double(), src is tgt, "field"))
        return sums
    src, tgt, x = _inputs(case, seed)
    if len(src) * len(tgt) > {"gradient": 1e10, "loss": 2e10}.get(entry, 8e10):
        return None
    same, x = src is tgt, x.double()
    if entry == "adjoint":
        return _direct(src, tgt, x, same, "field")
    if entry == "gradient":
        return _direct(tgt, src, x, same, "gradient")
    if entry == "loss":
        dtype = torch.float32
        measured = _direct(tgt, src, _normal(x.shape, 100 * seed + 60, dtype).double(), same, "field")
        residual = _direct(tgt, src, x, same, "field") - measured
        g = _direct(tgt, src, x, same, "gradient")
        full = torch.stack([g[..., [0, 1, 2]], g[..., [1, 3, 4]], g[..., [2, 4, 5]]], dim=-2)
        return {"moments": _direct(src, tgt, residual, same, "field"),
                "targets": (full * residual[:, :, None, :]).sum(dim=-1).sum(dim=0)}
    if entry in ("both", "host"):
        y = _direct(tgt, src, x[None] if entry == "host" else x, same, "both")
        h, phi = y[..., :3].contiguous(), y[..., 3].contiguous()
        return {"H": h[0], "phi": phi[0]} if entry == "host" else {"H": h, "phi": phi}
    return _direct(tgt, src, x, same, "field")


if __name__ == "__main__":  # the listed cases and a few drawn ones
    for c in listed() + [draw(random.Random(i)) for i in range(8)]:
        print(c)
