"""The benchmark shapes on the GPU against the reference's own outputs.

Fixtures (tests/golden/, written by make_golden.py from the reference FMM):
  * sphere_200k_p16  — the large-surface shape: two sphere surfaces, standard
    normal charges, p = 16, leaf capacity 128;
  * batch256_23_p12  — problem 23 of the 256-problem batch (clusters, cap 64, p = 12);
  * uniform_2m_p10, uniform_4m_p10_pot, plummer_2m_p12 — the largest sizes at
    which the reference evaluates the 4M-uniform and 16M-Plummer shapes;
  * selfgen_6k_p6    — a custom self generator with near and far pairs.
FP64 is held to 1e-12 relative L2 against the reference (the potential+gradient
fixtures are also covered, full/far/near, by test_gpu_parity.py).  The fixtures that
carry an FP64 direct sum also carry the reference's own error against it.  The
mixed path (M2L as split f16 products with FP32 accumulation, 22-bit operands;
FP32 pair arithmetic on FP64 coordinate differences) differs from FP64 by at
most the truncation error of order p (the reference's own error against the
direct sum), or by MIXED_ROUNDING where the truncation error is smaller than
what 22-bit operands carry; its error against the direct sum is at most the
reference's plus that bound.
"""
# the rounding of the mixed path, relative L2 against FP64: the operands of the
# f16 products carry 22 bits (2^-22 = 2.4e-7); measured 0.6-5.1e-7
MIXED_ROUNDING = 5e-7
import numpy as np
import pytest

from simplefmm_amd import api, workloads as W
from tests.helpers import golden_cases, golden_self_lists, load_golden, rel_l2

pytestmark = pytest.mark.gpu

PARITY = 1e-12
DIRECT = [c for c in golden_cases(None) if "reference_error_vs_direct" in load_golden(c)[0]]


def _plan(meta, pos, **kw):
    part = api.OctreePartitioner(pos, api.Box(pos)).refine(meta["max_level"], meta["cap"])
    assert part.level() == meta["depth"]
    return part, api.FMM3D(part, meta["p"], **kw)


@pytest.mark.parametrize("m2l_kernel", [0, 1], ids=["mfma", "rows"])
@pytest.mark.parametrize("case", ["sphere_200k_p16", "batch256_23_p12"])
def test_benchmark_shapes_match_reference(case, m2l_kernel):
    meta, g, pos, q = load_golden(case)
    print(f"case {case} n={meta['n']} p={meta['p']} cap={meta['cap']} m2l_kernel={m2l_kernel}", flush=True)
    _, fmm = _plan(meta, pos, ncharge=1, m2l_kernel=m2l_kernel)
    U = np.zeros((meta["n"], 4))
    fmm.rinv_potgrad(q, U)
    idx = g["idx"]
    assert rel_l2(U[idx, 0], g["phi_full"]) < PARITY
    assert rel_l2(U[idx, 1:], g["grad_full"]) < PARITY


@pytest.mark.parametrize("case", golden_cases("potential"))
def test_potential_only_matches_reference(case):
    meta, g, pos, q = load_golden(case)
    print(f"case {case} n={meta['n']} p={meta['p']}", flush=True)
    _, fmm = _plan(meta, pos, ncharge=1)
    U = np.zeros((meta["n"], 1))
    fmm.rinv(q, U)
    assert rel_l2(U[g["idx"], 0], g["phi_full"]) < PARITY


@pytest.mark.parametrize("m2l_kernel", [0, 1], ids=["mfma", "rows"])
def test_self_generator_matches_reference(m2l_kernel):
    meta, g, pos, q = load_golden("selfgen_6k_p6")
    lists = golden_self_lists(meta, pos)
    _, fmm = _plan(meta, pos, ncharge=1, m2l_kernel=m2l_kernel, self_lists=lists)
    idx = g["idx"]
    for which, suffix in ((api.BOTH, "full"), (api.FAR, "far"), (api.NEAR, "near")):
        U = np.zeros((meta["n"], 4))
        fmm.rinv_potgrad(q, U, which | api.SELF_LIST)
        assert rel_l2(U[idx, 0], g[f"phi_{suffix}"]) < PARITY, suffix
        assert rel_l2(U[idx, 1:], g[f"grad_{suffix}"]) < PARITY, suffix


def _direct_errors(meta, g, U):
    idx = g["idx"]
    err = {"phi": rel_l2(U[idx, 0], g["phi_direct"])}
    if "grad_direct" in g and U.shape[1] == 4:
        err["grad"] = rel_l2(U[idx, 1:], g["grad_direct"])
    return err


@pytest.mark.parametrize("case", DIRECT)
def test_fp64_error_equals_reference_error(case):
    # the GPU's FP64 error against the direct sum is the reference's own
    meta, g, pos, q = load_golden(case)
    print(f"case {case} n={meta['n']} p={meta['p']}", flush=True)
    _, fmm = _plan(meta, pos, ncharge=1)
    pot = meta["mode"] == "potential"
    U = np.zeros((meta["n"], 1 if pot else 4))
    fmm.rinv(q, U) if pot else fmm.rinv_potgrad(q, U)
    ref = meta["reference_error_vs_direct"]
    for k, v in _direct_errors(meta, g, U).items():
        print(f"  fp64 {k}: {v:.4e} (reference {ref[k]:.4e})", flush=True)
        assert abs(v - ref[k]) <= 1e-3 * ref[k]


@pytest.mark.parametrize("case", DIRECT)
def test_mixed_error_against_direct_sum(case):
    # the mixed path differs from FP64 by its rounding bound, and its error against
    # the direct sum is the reference's (the truncation error of order p) plus at
    # most that
    meta, g, pos, q = load_golden(case)
    print(f"case {case} n={meta['n']} p={meta['p']} mixed", flush=True)
    part, mixed = _plan(meta, pos, ncharge=1, precision=api.MIXED)
    fp64 = api.FMM3D(part, meta["p"], ncharge=1)
    pot = meta["mode"] == "potential"
    U = np.zeros((meta["n"], 1 if pot else 4))
    V = np.zeros_like(U)
    mixed.rinv(q, U) if pot else mixed.rinv_potgrad(q, U)
    fp64.rinv(q, V) if pot else fp64.rinv_potgrad(q, V)
    ref = meta["reference_error_vs_direct"]
    idx = g["idx"]
    for k, v in _direct_errors(meta, g, U).items():
        cols = slice(0, 1) if k == "phi" else slice(1, 4)
        diff = rel_l2(U[:, cols], V[:, cols])
        print(f"  mixed {k}: {v:.4e} against the direct sum (reference {ref[k]:.4e}); against FP64 {diff:.3e}",
              flush=True)
        bound = max(ref[k], MIXED_ROUNDING)
        assert diff <= bound, k
        assert v <= ref[k] + bound, k
    assert idx.size > 0


@pytest.mark.parametrize("prec", [api.FP64, api.MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("lone", [1, 3, 17, 64], ids=str)
def test_near_field_of_few_targets_beside_many_sources(lone, prec):
    # a few particles in coarse leaves next to a deep cluster: their near lists
    # are the whole cluster, cut into many runs, and a tail shorter than a tile
    rng = np.random.default_rng(lone)
    n = 30_011
    pos = np.concatenate([0.499 + 1e-3 * rng.uniform(size=(n - lone, 3)), rng.uniform(0.505, 1.0, (lone, 3))])
    box = api.Box(corner=[0.0, 0.0, 0.0], width=1.0)
    part = api.OctreePartitioner(pos, box).refine(20, 64)
    q = rng.uniform(-1, 1, n)
    U = np.zeros((n, 4))
    print(f"lone={lone} prec={prec} depth={part.level()}", flush=True)
    api.FMM3D(part, 4, ncharge=1, precision=prec).rinv_potgrad(q, U, api.NEAR)
    for i in list(range(n - lone, n))[:5] + [0, n // 2]:
        src = part.near_sources(i)
        src = src[src != i]
        d = pos[i] - pos[src]
        r = np.sqrt((d * d).sum(1))
        ref = np.array([(q[src] / r).sum(), *(-(q[src] / r**3) @ d)])
        # rounding: sums of |term| times a few units in the last place (FP32 pairs when mixed)
        scale = np.array([(np.abs(q[src]) / r).sum(), *((np.abs(q[src]) / r**3) @ np.abs(d))])
        assert np.all(np.abs(U[i] - ref) <= (1e-12 if prec == api.FP64 else 2e-6) * scale)


@pytest.mark.parametrize("p", [3, 12, 16])
@pytest.mark.parametrize("cells", [1, 768, 769], ids=["one", "last_split", "first_whole"])
def test_shifts_of_levels_around_the_split(cells, p):
    # `cells` refined nodes at level 4: 16/nc parents to a block, so 192 or 193
    # blocks of 4 components, where the M2M and L2L change from a workgroup per
    # child octant to one per block; children of some octants only
    rng = np.random.default_rng(cells)
    at = rng.permutation(16**3)[:cells]
    corner = np.stack([at // 256, at // 16 % 16, at % 16], 1)
    sub = rng.uniform(size=(cells, 5, 3))
    pos = np.concatenate([((corner[:, None, :] + sub) / 16).reshape(-1, 3), rng.uniform(size=(200, 3))])
    part = api.OctreePartitioner(pos, api.Box(corner=[0.0, 0.0, 0.0], width=1.0)).refine(20, 4)
    n = len(pos)
    q = rng.uniform(-1, 1, n)
    out = []
    for kernel in (0, 1):
        print(f"cells={cells} p={p} m2l_kernel={kernel} depth={part.level()}", flush=True)
        U = np.zeros((n, 4))
        api.FMM3D(part, p, ncharge=1, m2l_kernel=kernel).rinv_potgrad(q, U, api.FAR)
        out.append(U)
    # the same sums in another order: a few thousand terms, 1.1e-16 each
    assert rel_l2(out[0], out[1]) < 1e-13


@pytest.mark.parametrize("cells,p", [(4096, 8), (4097, 8), (4096, 16), (4097, 16)])
def test_shifts_of_a_level_around_1024_blocks(cells, p):
    # 4 parents to a block of 4 components: the L2L's change from p = 8 on, and at
    # p = 16 the M2M's chunk
    rng = np.random.default_rng(cells)
    at = rng.permutation(32**3)[:cells]
    corner = np.stack([at // 1024, at // 32 % 32, at % 32], 1)
    pos = ((corner[:, None, :] + rng.uniform(size=(cells, 5, 3))) / 32).reshape(-1, 3)
    part = api.OctreePartitioner(pos, api.Box(corner=[0.0, 0.0, 0.0], width=1.0)).refine(20, 4)
    q = rng.uniform(-1, 1, len(pos))
    out = []
    for kernel in (0, 1):
        print(f"cells={cells} p={p} m2l_kernel={kernel} depth={part.level()}", flush=True)
        U = np.zeros((len(pos), 4))
        api.FMM3D(part, p, ncharge=1, m2l_kernel=kernel).rinv_potgrad(q, U, api.FAR)
        out.append(U)
    # the same sums in another order: a few thousand terms, 1.1e-16 each
    assert rel_l2(out[0], out[1]) < 1e-13


@pytest.mark.parametrize("m2l_kernel,prec", [(0, api.FP64), (1, api.FP64), (0, api.MIXED)])
def test_stage_times_of_evaluations_with_and_without_a_far_field(m2l_kernel, prec):
    pos = np.random.default_rng(3).uniform(size=(20000, 3))
    part = api.OctreePartitioner(pos, api.Box(corner=[0.0, 0.0, 0.0], width=1.0)).refine(8, 40)
    fmm = api.FMM3D(part, 6, ncharge=1, m2l_kernel=m2l_kernel, precision=prec)
    q, U = np.ones(len(pos)), np.zeros((len(pos), 4))
    kinds = [api.BOTH, api.NEAR, api.FAR]
    fmm.record_stages(len(kinds))
    for which in kinds:
        fmm.rinv_potgrad(q, U, which)
    sets = fmm.recorded_stage_ms(8)
    assert len(sets) == len(kinds)
    fmm.record_stages(0)
    fmm.rinv_potgrad(q, U)
    for which, s in zip(kinds + [api.BOTH], sets + [fmm.stage_ms()]):
        print(which, s, flush=True)
        *stages, total = s.values()
        absent = [[], [1, 2, 3, 4, 5], [6]][kinds.index(which)]
        assert all((t == 0.0) == (k in absent) and t >= 0.0 for k, t in enumerate(stages))
        # each is a difference of clocks, rounded to single precision
        assert total == pytest.approx(sum(stages), rel=1e-5) and total < 1e3
