// FP64 M2L with one column per lane and the operators broadcast over 16-lane rows.
//
// FP64 vector and matrix arithmetic run at the same rate on gfx950 and share
// it (16x16x4 MFMA 76, v_fmac_f64 with a row broadcast 70 TFLOP/s measured; a
// wave of each together 72), so the M2L's cost is the multiply-adds it issues.
// The operators of rotate-translate-rotate (fmm.hpp:620-688) are blocks of
// every size 1..p+1: 16x16x4 tiles issue 1.9x the products the blocks hold at
// p = 12 (131 tiles of 1024 for 16 x 4407).  Here a lane holds one column (a
// target's source and a component), the products run as v_fmac_f64 at the
// blocks' own sizes, and the operator element comes from one lane of a
// register that a 16-lane row shares (DPP row_newbcast, the one DPP form of
// FP64): 16 elements to a register pair, so a wavefront keeps its share of the
// operators in registers and reloads it only when the polar class changes.
//
// A workgroup takes four rows.  A row is a block of 16/nc targets of one level
// and child octant (its lanes: target x component); the rows of a workgroup
// are the four octants of one z half under the same parents, whose
// interaction offsets fall into the same polar classes with the same counts.
// The workgroup walks steps, each of one polar class; a row has its own offset
// (azimuth) and sources in a step, so the rows need not have the same offsets.
// The columns' stage results lie in LDS as X[coefficient][lane]; a wavefront
// owns whole degrees (rotations) and whole orders (coaxial translation), each
// as its cos and sin blocks, and runs per step
//   1. azimuth e^{i m phi} of the gathered columns, forward rotation -> X rows
//      of its degrees; barrier;
//   2. coaxial translation of its orders, in place; barrier;
//   3. back rotation of its degrees, azimuth e^{-i m phi}, FP64 accumulators.
// Stage 3 of a step and stage 1 of the next touch the same wavefront's rows
// only, so two barriers per step suffice.  With order 0 divided by sqrt 2 the
// rotation is orthogonal and stage 3 uses stage 1's elements transposed.
// Columns and azimuths are requested a step ahead, operators a stage ahead.
//
// Measured (M2L stage, before: 16x16x4 MFMA pipeline, 46% matrix-core busy):
// 16M Plummer p = 12, 4 components 342 -> 175 ms; 2M Plummer 41.2 -> 21.6 ms;
// 100k uniform p = 8 0.95 -> 0.33 ms; 333k uniform p = 10, 3 components 8.6 ->
// 3.3 ms; 200k Plummer p = 12, 1 component 1.52 -> 0.88 ms; 200k on spheres p = 16
// (before: one offset at a time, four barriers) 5.03 -> 1.86 ms.  Bound by FP64
// issue (vector ALU busy 64% of the kernel at p = 12; two wavefronts of a SIMD
// reach 80%); the rest is waits at the two barriers and for the columns.
// Registers spilled per lane: p = 12 3, p = 13 48-63, p = 15 9-12 and p = 16 69-93 in
// the cos kernel (0 and 7-11 in the sin kernel), none at the other orders.
#pragma once

#include <cstddef>
#include <cstdint>
#include <type_traits>

#if defined(__HIPCC__)
#define SFMM_BC_HD __host__ __device__
#else
#define SFMM_BC_HD
#endif

namespace sfmm {

constexpr int kBcastMaxP = 16;

// Which blocks a kernel runs: both parts, or (two kernels, the second adding to
// the first's result) the cos and the sin blocks.  The parts meet only in the
// azimuths, so they can run apart; both gather all columns then.  Above p = 13 one
// kernel for both would exceed the registers and the instruction cache
// (24 sum (n+1)^2 + n^2 bytes of products; 64 KB shared by two compute units).  At
// p = 13 two kernels gain with several components and lose with one, whose columns
// cost most (200k Plummer, one kernel / two: 4 components 3.54 / 2.99 ms, 1 component
// 1.08 / 1.29).
enum BcastPart : int { kBcastBoth = 0, kBcastCos = 1, kBcastSin = 2 };
SFMM_BC_HD constexpr bool bcast_parted(int P) { return P > 13; }
SFMM_BC_HD constexpr bool bcast_runs_part(int mode, int part)  // part 0 = cos, 1 = sin
{
    return mode == kBcastBoth || mode == (part == 0 ? kBcastCos : kBcastSin);
}
// Rows of X.
SFMM_BC_HD constexpr int bcast_rows(int P, int mode)
{
    return mode == kBcastBoth ? (P + 1) * (P + 1) : mode == kBcastCos ? (P + 1) * (P + 2) / 2 : P * (P + 1) / 2;
}

// Wavefronts per workgroup and, as the register bound, per SIMD: a wavefront's
// registers hold its share of the operators (2 x 3 sum (n+1)^2 + n^2 doubles /
// 16 / waves), and 8 registers per gathered pair; X takes 512 (p+1)^2 bytes.  One FP64
// instruction stream issues every 6 clocks, two together every 5, three every
// 4.7, so the orders that fit take three wavefronts of a SIMD or more, from
// several workgroups; p = 9, 10 two workgroups of four; above, one of eight.
SFMM_BC_HD constexpr int bcast_waves(int P) { return P <= 5 ? 2 : (P <= 10 ? 4 : 8); }
SFMM_BC_HD constexpr int bcast_simd_waves(int P) { return P <= 4 ? 4 : (P <= 8 ? 3 : 2); }

// Work of a wavefront in one kind of stage: blocks (index, part), part 0 = cos,
// 1 = sin.  Rotations: index = degree n, block size n + 1 (cos) or n (sin).
// Coaxial: index = order m, block size p + 1 - m for either part (none of sin for m = 0).
struct BcastUnits {
    int count[8] = {};
    int idx[8][20] = {};
    int part[8][20] = {};
    SFMM_BC_HD constexpr bool has(int w, int i, int pt) const
    {
        for (int q = 0; q < count[w]; ++q)
            if (idx[w][q] == i && part[w][q] == pt) return true;
        return false;
    }
};

SFMM_BC_HD constexpr int bcast_size(int P, bool coax, int i, int part)
{
    return coax ? (part == 1 && i == 0 ? 0 : P + 1 - i) : (part == 0 ? i + 1 : i);
}

// Assignment of the blocks to the wavefronts: the cos and sin blocks of one
// index stay together (they share columns and accumulators, or operators)
// unless the pair exceeds a wavefront's share by a tenth; longest first, then
// moves and swaps that lower the largest load of a SIMD (wavefronts w, w + 4, ..),
// of a wavefront, and its registers for columns, weighed 20 : 15 : 3 (the loads of
// wavefronts alone: 1M Plummer p = 12 11.04 -> 11.12 ms, p = 11 9.05 -> 9.23, 300k p = 6
// 0.612 -> 0.620, 200k uniform p = 10 curl 0.472 -> 0.481).
SFMM_BC_HD constexpr BcastUnits bcast_units(int P, bool coax, int mode)
{
    const int NW = bcast_waves(P), NS = NW < 4 ? NW : 4;
    auto cost = [&](int i, int part) {
        const int s = bcast_runs_part(mode, part) ? bcast_size(P, coax, i, part) : 0;
        return s == 0 ? 0 : (coax ? s * s + 2 * s : 2 * s * s + 7 * s);
    };
    int total = 0;
    for (int i = 0; i <= P; ++i) total += cost(i, 0) + cost(i, 1);
    struct Item {
        int i = 0, parts = 0, cost = 0, cols = 0, w = 0;
    };
    Item it[40] = {};
    int ni = 0, cols = 0;
    for (int i = 0; i <= P; ++i) {
        const int c0 = cost(i, 0), c1 = cost(i, 1);
        const bool split = c0 > 0 && c1 > 0 && 10 * (c0 + c1) * NW > 11 * total;
        const int nc = bcast_size(P, coax, i, 0), parts = (c0 > 0 ? 1 : 0) | (c1 > 0 ? 2 : 0);
        if (parts == 0) continue;
        it[ni++] = Item{i, split ? 1 : parts, split ? c0 : c0 + c1, nc, 0};
        if (split) it[ni++] = Item{i, 2, c1, nc, 0};
        cols += split ? 2 * nc : nc;
    }
    for (int k = 1; k < ni; ++k)  // by cost, largest first
        for (int q = k; q > 0 && it[q].cost > it[q - 1].cost; --q) {
            const Item x = it[q];
            it[q] = it[q - 1];
            it[q - 1] = x;
        }
    auto score = [&](int placed) {
        int load[8] = {}, simd[4] = {}, nc[8] = {};
        for (int k = 0; k < placed; ++k) {
            load[it[k].w] += it[k].cost;
            simd[it[k].w % NS] += it[k].cost;
            nc[it[k].w] += it[k].cols;
        }
        // relative squares, so that every load above the mean counts
        int64_t ll = 0, ss = 0, cc = 0;
        for (int w = 0; w < NW; ++w) {
            ll += static_cast<int64_t>(load[w]) * load[w];
            cc += static_cast<int64_t>(nc[w]) * nc[w];
            if (w < NS) ss += static_cast<int64_t>(simd[w]) * simd[w];
        }
        const int64_t tt = static_cast<int64_t>(total) * total;
        return 400000000 * ss / tt * NS + 300000000 * ll / tt * NW +
               (coax ? 0 : 60000000 * cc / (static_cast<int64_t>(cols) * cols) * NW);
    };
    for (int k = 0; k < ni; ++k) {
        int best = 0;
        int64_t bs = int64_t(1) << 60;
        for (int w = 0; w < NW; ++w) {
            it[k].w = w;
            const int64_t sc = score(k + 1);
            if (sc < bs) bs = sc, best = w;
        }
        it[k].w = best;
    }
    int64_t now = score(ni);
    for (bool better = true; better;) {
        better = false;
        for (int k = 0; k < ni; ++k) {
            for (int w = 0; w < NW; ++w) {
                const int old = it[k].w;
                it[k].w = w;
                const int64_t sc = score(ni);
                if (sc < now) now = sc, better = true;
                else it[k].w = old;
            }
            for (int q = 0; q < k; ++q) {
                const int wk = it[k].w, wq = it[q].w;
                it[k].w = wq, it[q].w = wk;
                const int64_t sc = score(ni);
                if (sc < now) now = sc, better = true;
                else it[k].w = wk, it[q].w = wq;
            }
        }
    }
    BcastUnits u;
    for (int k = 0; k < ni; ++k)
        for (int part = 0; part < 2; ++part)
            if (it[k].parts >> part & 1) {
                const int w = it[k].w;
                u.idx[w][u.count[w]] = it[k].i;
                u.part[w][u.count[w]] = part;
                ++u.count[w];
            }
    return u;
}

// First operator element of the wavefront's block q, and all its elements (q = count).
// Coaxial cos and sin of one order in one wavefront share their elements.
SFMM_BC_HD constexpr int bcast_elem(int P, const BcastUnits& u, bool coax, int w, int q)
{
    int e = 0;
    for (int k = 0; k < q; ++k) {
        bool again = false;
        for (int j = 0; j < k; ++j) again = again || (coax && u.idx[w][j] == u.idx[w][k]);
        const int s = bcast_size(P, coax, u.idx[w][k], u.part[w][k]);
        if (!again) e += s * s;
    }
    return e;
}
SFMM_BC_HD constexpr int bcast_block(int P, const BcastUnits& u, bool coax, int w, int q)
{
    if (coax)
        for (int j = 0; j < q; ++j)
            if (u.idx[w][j] == u.idx[w][q]) return bcast_elem(P, u, coax, w, j);
    return bcast_elem(P, u, coax, w, q);
}
SFMM_BC_HD constexpr int bcast_regs(int P, const BcastUnits& u, bool coax, int w)
{
    return (bcast_elem(P, u, coax, w, u.count[w]) + 15) / 16;
}
// Registers of all wavefronts before w (w = waves: of one operator).
SFMM_BC_HD constexpr int bcast_reg0(int P, const BcastUnits& u, bool coax, int w)
{
    int r = 0;
    for (int k = 0; k < w; ++k) r += bcast_regs(P, u, coax, k);
    return r;
}

// Workgroups a compute unit holds at once (LDS and wavefronts).
SFMM_BC_HD constexpr int bcast_resident(int P)
{
    const int lds = 160 * 1024 / (512 * bcast_rows(P, bcast_parted(P) ? kBcastCos : kBcastBoth)), wv = 4 * bcast_simd_waves(P) / bcast_waves(P);
    return lds < wv ? lds : wv;
}

// Length of the next run when `left` steps of an XCD's share are still to be
// dealt out: whole groups (up to 189 steps) while there are many left, then ever
// shorter runs, so that the last workgroups end together.  A run's partial
// sums cost about 3 steps to write and add, hence the least length, less where even
// all steps are few (M2L with least 2 / 4 / 8 / 16 steps, us: 2k uniform p = 8 34.6 / 26.9
// / 29.2 / 41.1; 5k Plummer p = 8 63.4 / 50.5 / 47.8 / 62.0; 20k uniform p = 8 80.8 /
// 70.9 / 65.5 / 64.4; 20k Plummer p = 12 322 / 313 / 303 / 315).
inline int64_t bcast_run_steps(int P, int64_t left, int64_t n_step)
{
    const int64_t r = left * 2 / (3 * 32 * bcast_resident(P)), least = n_step < 2048 ? 4 : 8;
    return r < least ? least : r;
}

SFMM_BC_HD constexpr int bcast_pairs(int P) { return (P + 1) * (P + 2) / 2; }
SFMM_BC_HD constexpr int bcast_pair(int n, int m) { return n * (n + 1) / 2 + m; }

}  // namespace sfmm
