"""The evaluations whose speed this framework is measured by.

A case is one call (or the calls of one step) of a program that holds a built
tree and plan: charges in, potentials and gradients out, accumulated into a
zeroed output array, through the public binding (`simplefmm_amd.api`).  The
listed cases are the shapes of the repository's fixtures and benchmark, from a
few thousand points, where launches and latency count, to the 16M-point Plummer
sphere of `bench.py`; `draw` gives others of the same ranges.

Fields of a case:
  call   "device": arrays in HBM, asynchronous on the plan's stream
         "host":   numpy arrays through the reference's rinv interface
         "batch":  independent problems in one batch launch
  gen    point distribution (`simplefmm_amd.workloads`, made here on the GPU)
  n, p, cap, mixed    points, expansion order, leaf capacity, precision
  kind   "pot1", "pot3" (potentials of 1 or 3 charges), "curl" (vector charges,
         rinv<true>), "potgrad" (scalar charge, phi and grad phi),
         "both" (host only: rinv and rinv<true> of vector charges, main.cpp's pair)
  which  "both", "far" (rinv_nonear) or "near" (N2N)
  count, nmax   (batch) problems, sizes log-uniform in [10_000, nmax], p from 6, 8, 10, 12
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from simplefmm_amd import api

KINDS = {"pot1": (api.POTENTIAL, 1, 1, 1), "pot3": (api.POTENTIAL, 3, 3, 3), "curl": (api.CURL, 3, 3, 3),
         "potgrad": (api.POTGRAD, 1, 1, 4)}  # kind, ncharge, charges and outputs per point
WHICH = {"both": api.BOTH, "far": api.FAR, "near": api.NEAR}
EXACT_PAIRS = 8e10  # the direct sum is taken up to this many pairs


def _device(name, gen, n, p, cap, kind="potgrad", mixed=False, which="both", call="device"):
    return {"name": name, "call": call, "gen": gen, "n": n, "p": p, "cap": cap, "kind": kind, "mixed": mixed,
            "which": which}


def listed():
    return [
        # a small system inside a larger program's loop: launches and latency
        _device("uniform_2k_p8", "uniform", 2000, 8, 64),
        # the reference driver's pair of calls, rinv and rinv<true> of vector charges, on host arrays
        _device("vector_5k_p8_host", "uniform", 5000, 8, 64, kind="both", call="host"),
        # a small adaptive tree with the mixed path
        _device("plummer_20k_p12_mixed", "plummer", 20_000, 12, 64, mixed=True),
        # the medium uniform system of the benchmark, plain FP64
        _device("uniform_100k_p8", "uniform", 100_000, 8, 64),
        # potentials alone (one component per node)
        _device("plummer_200k_p12_pot", "plummer", 200_000, 12, 64, kind="pot1"),
        # vector charges to a vector field (three components); a ragged size
        _device("vector_333331_p10_curl", "uniform", 333_331, 10, 64, kind="curl"),
        # points on surfaces at the highest order
        _device("sphere_200k_p16", "sphere", 200_000, 16, 128),
        # independent cluster problems of four orders in one launch
        {"name": "batch16_clusters", "call": "batch", "count": 16, "nmax": 300_000, "cap": 64, "mixed": False},
        # an N-body step's size, FP64
        _device("plummer_2m_p12", "plummer", 2_000_000, 12, 64),
        # the large uniform system, mixed
        _device("uniform_4m_p10_mixed", "uniform", 1 << 22, 10, 64, mixed=True),
        # the headline workload, mixed and FP64
        _device("plummer_16m_p12_mixed", "plummer", 1 << 24, 12, 64, mixed=True),
        _device("plummer_16m_p12", "plummer", 1 << 24, 12, 64),
    ]


def draw(rng: random.Random):
    if rng.random() < 0.1:
        return {"call": "batch", "count": rng.randrange(4, 25), "nmax": rng.randrange(20_000, 400_000),
                "cap": rng.choice([32, 64]), "mixed": rng.random() < 0.3}
    n = int(round(math.exp(rng.uniform(math.log(1500), math.log(4.2e6)))))
    p = rng.choice([4, 6, 7, 8, 8, 9, 10, 10, 11, 12, 12, 12, 16])
    mixed = rng.random() < 0.35
    kind = rng.choice(["pot1", "pot3", "curl", "potgrad", "potgrad", "potgrad"])
    which = rng.choice(["both"] * 8 + ["far", "near"])
    call = "device"
    if n < 300_000 and rng.random() < 0.25:
        call, which = "host", "both"
        kind = rng.choice([kind, "both"])
    gen = rng.choice(["uniform", "plummer", "clusters", "sphere"])
    return {"call": call, "gen": gen, "n": n, "p": p, "cap": rng.choice([32, 64, 64, 64, 100, 128]), "kind": kind,
            "mixed": mixed, "which": which}


# ------------------------------------------------------------------ inputs
def _rand(g, *shape):
    return torch.rand(*shape, generator=g, dtype=torch.float64, device=g.device)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, dtype=torch.float64, device=g.device)


def _points(gen, n, g):
    """The distributions of simplefmm_amd.workloads, drawn on the GPU."""
    if gen == "uniform":
        return _rand(g, n, 3)
    if gen == "plummer":  # scale radius 1, truncated at 50
        mmax = 50.0 ** 3 / (1.0 + 50.0 * 50.0) ** 1.5
        r = 1.0 / torch.sqrt(((1.0 - _rand(g, n)) * mmax) ** (-2.0 / 3.0) - 1.0)
        c = 2.0 * _rand(g, n) - 1.0
        phi = 2.0 * math.pi * _rand(g, n)
        s = torch.sqrt(torch.clamp(1.0 - c * c, min=0.0))
        return torch.stack([r * s * torch.cos(phi), r * s * torch.sin(phi), r * c], 1)
    if gen == "clusters":  # up to 8 isotropic clusters in the unit cube
        k = 1 + int(torch.randint(0, 8, (1,), generator=g, device=g.device))
        centre, sigma = _rand(g, k, 3), 0.02 + 0.18 * _rand(g, k)
        got, have = [], 0
        while have < n:
            m = 2 * (n - have) + 64
            w = torch.randint(0, k, (m,), generator=g, device=g.device)
            x = centre[w] + sigma[w, None] * _randn(g, m, 3)
            x = x[((x >= 0) & (x < 1)).all(1)][: n - have]
            got.append(x)
            have += len(x)
        return torch.cat(got)
    x = _randn(g, n, 3)  # "sphere": the unit sphere, a tenth on a sphere of radius 1/2
    x /= x.norm(dim=1, keepdim=True)
    x[n - int(round(0.1 * n)):] *= 0.5
    return x


def _charges(gen, n, nq, g):
    if gen == "plummer":
        return 1.0 - _rand(g, n, nq)  # masses in (0, 1]
    return _randn(g, n, nq) if gen == "sphere" else 2.0 * _rand(g, n, nq) - 1.0


def _inputs(case, seed):
    """(positions, charges) as torch tensors; of a batch, a list of (p, positions, charges)."""
    g = torch.Generator(device="cuda" if torch.cuda.is_available() else "cpu")
    g.manual_seed(seed)
    if case["call"] == "batch":
        r, out = random.Random(1000 * case["count"] + case["nmax"]), []  # the sizes are the case's own
        for _ in range(case["count"]):
            n = int(round(math.exp(r.uniform(math.log(10_000), math.log(case["nmax"])))))
            p = r.choice([6, 8, 10, 12])
            out.append((p, _points("clusters", n, g), _charges("clusters", n, 1, g)))
        return out
    nq = 3 if case["kind"] == "both" else KINDS[case["kind"]][2]
    return _points(case["gen"], case["n"], g), _charges(case["gen"], case["n"], nq, g)


def _plan(pos, p, cap, mixed, ncharge):
    x = pos.cpu().numpy()
    # large trees are built on the GPU, as bench.py builds them
    tree = api.OctreePartitioner(x, api.Box(x)).refine(20, cap, on_device=len(x) >= 1_000_000)
    return api.FMM3D(tree, p, ncharge=ncharge, precision=api.MIXED if mixed else api.FP64)


def prepare(case, seed):
    if case["call"] == "batch":
        probs, items = [], []
        for p, pos, q in _inputs(case, seed):
            fmm = _plan(pos, p, case["cap"], case["mixed"], 1)
            u = torch.zeros(len(pos), 4, dtype=torch.float64, device="cuda")
            probs.append({"fmm": fmm, "q": q, "u": u})
            items.append((fmm, api.POTGRAD, 1, q.data_ptr(), u.data_ptr()))
        torch.cuda.synchronize()
        return {"case": case, "probs": probs, "batch": api.Batch(items, streams=4), "stream": torch.cuda.Stream()}
    pos, q = _inputs(case, seed)
    fmm = _plan(pos, case["p"], case["cap"], case["mixed"], q.shape[1])
    if case["call"] == "host":
        nout = 6 if case["kind"] == "both" else KINDS[case["kind"]][3]
        shapes = [3, 3] if nout == 6 else [nout]
        return {"case": case, "fmm": fmm, "q": q.cpu().numpy(), "u": [np.zeros((len(pos), k)) for k in shapes]}
    u = torch.zeros(case["n"], KINDS[case["kind"]][3], dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()  # the plan's stream does not wait for torch's
    return {"case": case, "fmm": fmm, "q": q, "u": u, "stream": torch.cuda.ExternalStream(fmm.stream())}


def run(state):
    case = state["case"]
    if case["call"] == "batch":
        with torch.cuda.stream(state["stream"]):
            for pb in state["probs"]:
                pb["u"].zero_()
        state["batch"].launch(state["stream"].cuda_stream)
        return [pb["u"] for pb in state["probs"]]
    fmm, q = state["fmm"], state["q"]
    if case["call"] == "host":
        for u in state["u"]:
            u[:] = 0.0
        if case["kind"] == "potgrad":
            fmm.rinv_potgrad(q, state["u"][0])
        elif case["kind"] == "both":
            fmm.rinv(q, state["u"][0])
            fmm.rinv(q, state["u"][1], gradient=True)
        else:
            fmm.rinv(q, state["u"][0], gradient=case["kind"] == "curl")
        return state["u"]
    kind, nq = KINDS[case["kind"]][:2]
    with torch.cuda.stream(state["stream"]):
        state["u"].zero_()
    fmm.evaluate_device(kind, nq, q.data_ptr(), state["u"].data_ptr(), WHICH[case["which"]])
    return state["u"]


# ------------------------------------------------------------------ what a pass cannot do without
def _work(n, p, cap, nq, nout, which, nexp):
    """Estimates from the shape alone: leaves 0.4 full, 8/7 nodes per leaf, 170
    interactions per node, 27 neighbour leaves."""
    leaves = max(1.0, n / (0.4 * cap))
    mac = sum((i + 1) ** 2 + i * i for i in range(p + 1))
    K = (p + 1) ** 2
    flops = 0.0
    if which != "near":
        flops += leaves * 8 / 7 * 170 * nexp * 2 * (3 * mac + 4 * p * (p + 1))  # M2L, rotate-translate-rotate
        flops += n * K * (6 + 4 * nexp) * 2                                    # P2M, L2P
    if which != "far":
        flops += n * 27 * 0.4 * cap * (12 + 2 * nout)
    return {"bytes": 8.0 * n * (3 + nq + nout), "flops": flops}


def work(case):
    if case["call"] == "batch":
        parts, r = [], random.Random(1000 * case["count"] + case["nmax"])
        for _ in range(case["count"]):
            n = int(round(math.exp(r.uniform(math.log(10_000), math.log(case["nmax"])))))
            parts.append(_work(n, r.choice([6, 8, 10, 12]), case["cap"], 1, 4, "both", 4))
        return {k: sum(w[k] for w in parts) for k in ("bytes", "flops")}
    if case["kind"] == "both":
        w = _work(case["n"], case["p"], case["cap"], 3, 3, case["which"], 3)
        return {k: 2 * v for k, v in w.items()}
    nq, nout = KINDS[case["kind"]][2:]
    return _work(case["n"], case["p"], case["cap"], nq, nout, case["which"], nout)


# ------------------------------------------------------------------ the direct sum
def _direct(kind, pos, q):
    n = len(pos)
    nout = KINDS[kind][3]
    out = torch.empty(n, nout, dtype=torch.float64, device=pos.device)
    step = max(1, min(n, 40_000_000 // n))
    for a in range(0, n, step):
        b = min(n, a + step)
        d = [pos[a:b, None, k] - pos[None, :, k] for k in range(3)]  # x_i - x_j
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        own = torch.arange(a, b, device=pos.device)
        r2[own - a, own] = math.inf
        rinv = torch.rsqrt(r2)
        if kind in ("pot1", "pot3"):
            out[a:b] = rinv @ q
            continue
        r3 = rinv * rinv * rinv
        if kind == "potgrad":
            out[a:b, 0] = rinv @ q[:, 0]
            for k in range(3):
                out[a:b, 1 + k] = -((d[k] * r3) @ q[:, 0])
        else:  # sum Q_j x (x_i - x_j) / r^3
            m = [(d[k] * r3) @ q for k in range(3)]  # [k][:, c] = sum Q_c d_k / r^3
            out[a:b, 0] = m[2][:, 1] - m[1][:, 2]
            out[a:b, 1] = m[0][:, 2] - m[2][:, 0]
            out[a:b, 2] = m[1][:, 0] - m[0][:, 1]
    return out


def exact(case, seed):
    """The direct sum, where it is short enough; the far or near part alone has none."""
    if case["call"] == "batch":
        left, out = EXACT_PAIRS, []
        for _, pos, q in _inputs(case, seed):
            left -= float(len(pos)) ** 2
            out.append(_direct("potgrad", pos, q) if left >= 0 else None)
        return out
    if case["which"] != "both" or float(case["n"]) ** 2 > EXACT_PAIRS:
        return None
    pos, q = _inputs(case, seed)
    kinds = ["pot3", "curl"] if case["kind"] == "both" else [case["kind"]]
    out = [_direct(k, pos, q) for k in kinds]
    return out if case["call"] == "host" else out[0]
