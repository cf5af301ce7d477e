"""Device memory of FP64 plans: what an evaluation's expansions take, and evaluations
where memory is short (SFMM_FAULT_ALLOC_BYTES fails every larger allocation)."""
import numpy as np
import pytest

from simplefmm_amd import api, workloads as W
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu

# the order of a few hundred additions per coefficient differs
TOLERANCE = 1e-13


def _expansions(part, p, nc):
    """Bytes of the nodes' nc expansions in FP64."""
    return 8 * nc * (p + 1) ** 2 * part.info().n_node


def test_expansions_take_two_arrays():
    # the multipoles (whose place the local expansions take) and the M2L's copy of
    # them, (p + 2) / (p + 1) as large; work lists of at most 343 steps of 80 bytes
    # per 16 nodes (1.7 of a node's 5.4 kB); partial sums and particles below 0.3 GB
    import torch
    n, p = 2_000_000, 12
    pos, q = W.plummer(n, seed=41)
    part = api.OctreePartitioner(pos, api.Box(pos)).refine(20, 64, on_device=True)
    fmm = api.FMM3D(part, p, ncharge=1)
    dq = torch.from_numpy(q).cuda()
    du = torch.zeros((n, 4), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    fmm.evaluate_device(api.POTGRAD, 1, dq.data_ptr(), du.data_ptr())
    fmm.synchronize()
    used, M = before - torch.cuda.mem_get_info()[0], _expansions(part, p, 4)
    print(f"n={n} p={p}: {used / 1e9:.2f} GB, multipoles {M / 1e9:.2f} GB", flush=True)
    assert used < (1 + 14 / 13 + 0.32) * M + 0.3e9


KINDS = {"potgrad": (api.POTGRAD, 1, 4), "potential": (api.POTENTIAL, 1, 1), "curl": (api.CURL, 3, 3)}


# (a target's work list, 0.8-1.1 kB, has to be smaller than its multipoles)
@pytest.mark.parametrize("gen,n,cap,p,kinds", [
    ("uniform_cube", 30_000, 32, 8, "potgrad"), ("uniform_cube", 30_000, 32, 8, "curl"),
    ("uniform_cube", 40_000, 64, 6, "potgrad"), ("sphere_shell", 20_000, 16, 12, "potgrad"),
    ("sphere_shell", 20_000, 16, 12, "potential"), ("pairs", 6_000, 1, 16, "potgrad"),
    ("pairs", 6_000, 1, 16, "potential"), ("uniform_cube", 600, 8, 16, "curl")])
def test_evaluations_where_no_allocation_exceeds_the_multipoles(gen, n, cap, p, kinds, monkeypatch):
    # the copy of the multipoles takes one level at a time, groups are not cut, and
    # (pairs: 3000 cells of two points, each in its own octant) the M2M's partial sums
    # of 188 blocks are made in pieces
    rng = np.random.default_rng(n)
    kind, nq, nout = KINDS[kinds]
    if gen == "pairs":
        at = rng.permutation(16**3)[: n // 2]
        cell = np.stack([at // 256, at // 16 % 16, at % 16], 1)
        pos = np.concatenate([cell + rng.uniform(0.05, 0.45, cell.shape), cell + rng.uniform(0.55, 0.95, cell.shape)]) / 16
        box = api.Box(corner=[0.0, 0.0, 0.0], width=1.0)
    else:
        pos, _ = getattr(W, gen)(n, seed=n)
        box = api.Box(pos)
    part = api.OctreePartitioner(pos, box).refine(20, cap)
    Q = rng.uniform(-1, 1, (n, nq))
    ref, u, again, free = (np.zeros((n, nout)) for _ in range(4))
    api.FMM3D(part, p, ncharge=nq)._eval(kind, nq, Q, ref, api.FAR)
    short = api.FMM3D(part, p, ncharge=nq)
    limit = _expansions(part, p, nout)
    print(f"{gen} n={n} p={p} kind={kind}: at most {limit} bytes", flush=True)
    monkeypatch.setenv("SFMM_FAULT_ALLOC_BYTES", str(limit))
    short._eval(kind, nq, Q, u, api.FAR)
    short._eval(kind, nq, Q, again, api.FAR)
    monkeypatch.delenv("SFMM_FAULT_ALLOC_BYTES")
    short._eval(kind, nq, Q, free, api.FAR)
    assert np.array_equal(u, again) and np.array_equal(u, free)
    assert rel_l2(u, ref) < TOLERANCE


def test_component_counts_before_and_after_memory_got_short(monkeypatch):
    # lists made for the copy of all levels are not used with the copy of one
    n, p = 20_000, 9
    pos, _ = W.plummer(n, seed=43)
    part = api.OctreePartitioner(pos, api.Box(pos)).refine(20, 32)
    rng = np.random.default_rng(4)
    cases = [(api.POTENTIAL, nq, rng.uniform(-1, 1, (n, nq))) for nq in (1, 2, 3, 4)]
    ref = []
    for kind, nq, Q in cases:
        ref.append(np.zeros((n, nq)))
        api.FMM3D(part, p, ncharge=4)._eval(kind, nq, Q, ref[-1], api.FAR)
    fmm = api.FMM3D(part, p, ncharge=4)
    for k in (0, 1, 3, 0, 2, 1):  # memory is short when four components come
        kind, nq, Q = cases[k]
        if k == 3:
            monkeypatch.setenv("SFMM_FAULT_ALLOC_BYTES", str(_expansions(part, p, 4)))
        u = np.zeros((n, nq))
        fmm._eval(kind, nq, Q, u, api.FAR)
        monkeypatch.delenv("SFMM_FAULT_ALLOC_BYTES", raising=False)
        print(f"n={n} p={p} ncharge={nq}: {rel_l2(u, ref[k]):.1e}", flush=True)
        assert rel_l2(u, ref[k]) < TOLERANCE


def test_near_field_of_fat_leaves_takes_no_more_partial_sums():
    # 1562 targets to a leaf: runs of 128 sources (2^18 pairs) and 191 runs to a leaf
    # on average, 32 bytes per target and run: 0.61 GB
    import torch
    n = 100_000
    rng = np.random.default_rng(7)
    pos, Q = rng.uniform(size=(n, 3)), rng.uniform(-1, 1, (n, 1))
    part = api.OctreePartitioner(pos, api.Box(corner=[0.0, 0.0, 0.0], width=1.0)).refine(20, 2000)
    fmm = api.FMM3D(part, 2, ncharge=1)
    dq = torch.from_numpy(Q).cuda()
    du = torch.zeros((n, 4), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    fmm.evaluate_device(api.POTGRAD, 1, dq.data_ptr(), du.data_ptr(), api.NEAR)
    fmm.synchronize()
    used = before - torch.cuda.mem_get_info()[0]
    print(f"n={n}: {used / 1e9:.2f} GB", flush=True)
    assert used < 0.7e9
    tg = np.arange(0, n, 997)
    got = du.cpu().numpy()
    for i in tg[:20]:
        src = part.near_sources(i)
        src = src[src != i]
        d = pos[i] - pos[src]
        r = np.sqrt((d * d).sum(1))
        scale = (np.abs(Q[src, 0]) / r).sum()
        assert abs(got[i, 0] - (Q[src, 0] / r).sum()) <= 1e-12 * scale
