"""The FP64 M2L with broadcast operators (simplefmm_amd/csrc/m2l_bcast.hpp).

On the CPU: every operator block is assigned to one wavefront, and the built
kernels keep two wait states between a vector write of a register and its read
through DPP (the products are inline assembly, which the compiler does not
check).  On the GPU: every order and component count against the row kernel
(m2l_kernel = 1), which shares only the operator tables with it.
"""
import os
import re
import shutil
import subprocess

import numpy as np
import pytest

from simplefmm_amd import api, workloads as W
from tests.helpers import rel_l2

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"

PROGRAM = r"""
#include "m2l_bcast.hpp"
#include <cstdio>
using namespace sfmm;
int main()
{
    for (int P = 1; P <= kBcastMaxP; ++P)
        for (int coax = 0; coax < 2; ++coax) {
          for (int mode = bcast_parted(P) ? 1 : 0; mode <= (bcast_parted(P) ? 2 : 0); ++mode) {
            const BcastUnits u = bcast_units(P, coax, mode);
            int seen[20][2] = {}, most = 0, total = 0;
            for (int w = 0; w < bcast_waves(P); ++w) {
                int cost = 0, last = -1;
                for (int q = 0; q < u.count[w]; ++q) {
                    const int s = bcast_size(P, coax, u.idx[w][q], u.part[w][q]);
                    ++seen[u.idx[w][q]][u.part[w][q]];
                    cost += s * s;
                    const int e = bcast_block(P, u, coax, w, q);
                    const bool shared = coax && q > 0 && u.idx[w][q] == u.idx[w][q - 1];
                    if (shared ? e != last : e < 0 || e + s * s > 16 * bcast_regs(P, u, coax, w)) return std::printf("FAIL elements P=%d\n", P);
                    last = e;
                }
                most = cost > most ? cost : most;
                total += cost;
            }
            for (int i = 0; i <= P; ++i)
                for (int part = 0; part < 2; ++part)
                    if (seen[i][part] != (bcast_runs_part(mode, part) && bcast_size(P, coax, i, part) > 0))
                        return std::printf("FAIL block %d %d P=%d coax=%d: %d times\n", i, part, P, coax, seen[i][part]);
            if (most * bcast_waves(P) > 2 * total) return std::printf("FAIL balance P=%d coax=%d\n", P, coax);
          }
        }
    std::printf("OK\n");
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_blocks_are_assigned_once(tmp_path):
    src = tmp_path / "units.cpp"
    src.write_text(PROGRAM)
    exe = str(tmp_path / "units")
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "simplefmm_amd", "csrc"), str(src), "-o", exe], check=True)
    assert subprocess.run([exe], capture_output=True, text=True).stdout.strip() == "OK"


def _registers(token):
    m = re.match(r"-?\|?v\[(\d+):(\d+)\]", token) or re.match(r"-?\|?v(\d+)", token)
    return set() if m is None else set(range(int(m[1]), int(m[m.lastindex]) + 1))


def dpp_hazards(listing):
    """(DPP reads, those within two wait states of a vector write of the register)."""
    reads, bad, recent = 0, [], []
    for line in listing:
        text = line.split("//")[0].strip()
        m = re.match(r"([a-z]+_\w+)\s*(.*)", text)
        if m is None:
            continue
        op, args = m[1], m[2].split(",")
        if "row_newbcast" in text:
            reads += 1
            src, waits = _registers(args[1].strip()), 0
            for wrote, states in reversed(recent):
                if waits >= 2:
                    break
                if wrote & src:
                    bad.append(text)
                    break
                waits += states
        wrote = _registers(args[0].strip()) if op.startswith("v_") and not op.startswith("v_cmp") else set()
        recent = recent[-3:] + [(wrote, int(args[0]) + 1 if op == "s_nop" else 1)]
    return reads, bad


def test_hazard_check_sees_a_planted_hazard():
    near = ["v_mov_b32_e32 v4, v9", "s_nop 0", "v_fmac_f64_dpp v[0:1], v[4:5], v[2:3] row_newbcast:3 row_mask:0xf"]
    far = [near[0], "s_nop 1", near[2]]
    assert len(dpp_hazards(near)[1]) == 1 and dpp_hazards(far) == (1, [])


@pytest.mark.skipif(not (os.path.exists(OBJDUMP) and os.path.exists(api.LIB_PATH)), reason="needs the built library")
def test_dpp_reads_wait_for_vector_writes(tmp_path):
    lib = shutil.copy(api.LIB_PATH, tmp_path / "libsfmm.so")
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
    reads = 0
    for name in sorted(os.listdir(tmp_path)):
        if "gfx950" not in name:
            continue
        out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(tmp_path / name)], check=True,
                             capture_output=True, text=True).stdout
        n, bad = dpp_hazards(out.splitlines())
        reads += n
        assert not bad, (name, bad[:3])
    assert reads > 10000


# the two kernels round in different orders: a few hundred additions per
# coefficient, each relative 1.1e-16
TOLERANCE = 1e-13


@pytest.mark.gpu
@pytest.mark.parametrize("p", range(1, 17))
@pytest.mark.parametrize("gen,n,cap", [("uniform_cube", 2500, 40), ("sphere_shell", 6000, 16), ("uniform_cube", 40, 1)],
                         ids=["ragged", "sparse", "deep"])
def test_matches_row_kernel(gen, n, cap, p):
    pos, _ = getattr(W, gen)(n, seed=p)
    part = api.OctreePartitioner(pos, api.Box(pos)).refine(20, cap)
    new = api.FMM3D(part, p, ncharge=4)
    old = api.FMM3D(part, p, ncharge=4, m2l_kernel=1)
    rng = np.random.default_rng(p)
    for kind, nq, nout in ((0, 4, 4), (0, 1, 1), (0, 2, 2), (0, 3, 3), (1, 3, 3), (2, 1, 4)):
        print(f"{gen} n={n} cap={cap} p={p} kind={kind} ncharge={nq}", flush=True)
        Q = rng.uniform(-1, 1, (n, nq))
        u, again, v = (np.zeros((n, nout)) for _ in range(3))
        new._eval(kind, nq, Q, u, api.FAR)
        new._eval(kind, nq, Q, again, api.FAR)
        old._eval(kind, nq, Q, v, api.FAR)
        assert np.array_equal(u, again)
        assert rel_l2(u, v) < TOLERANCE


@pytest.mark.gpu
@pytest.mark.parametrize("kind,nq,nout", [(2, 1, 4), (0, 1, 1)], ids=["potgrad", "potential"])
def test_whole_groups_and_runs_match_row_kernel(kind, nq, nout):
    # enough groups that the first stay whole and the last are cut into runs
    n, p = 150_000, 4
    pos, _ = W.uniform_cube(n, seed=2)
    part = api.OctreePartitioner(pos, api.Box(pos)).refine(20, 4)
    Q = np.random.default_rng(5).uniform(-1, 1, (n, nq))
    u, v = np.zeros((n, nout)), np.zeros((n, nout))
    print(f"n={n} p={p} kind={kind}", flush=True)
    api.FMM3D(part, p, ncharge=1)._eval(kind, nq, Q, u, api.FAR)
    api.FMM3D(part, p, ncharge=1, m2l_kernel=1)._eval(kind, nq, Q, v, api.FAR)
    assert rel_l2(u, v) < TOLERANCE
