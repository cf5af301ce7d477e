// M2L of the mixed-precision path on the f16 matrix cores, with hi/lo split
// products (Ootomo & Yokota, "Recovering single precision accuracy from Tensor
// Cores while surpassing the FP32 theoretical peak performance", IJHPCA 2022).
//
// The rotate-translate-rotate operator of fmm.hpp:620-688 for an offset d with
// azimuth phi, polar class c and distance |d| factors as
//     L~ += Az(-phi) D_c Az(phi) M~,
// where Az(phi) multiplies each coefficient of order m by e^{i m phi} and D_c =
// R_c^T T_|d| R_c (polar rotation, coaxial translation, back rotation) depends on
// the polar class only (|d| is fixed by it).  In the real form D_c is block
// diagonal: a cos block on the Re parts (m >= 0) and a sin block on the Im parts
// (m >= 1).  This kernel stores D_c densely (70 classes, level independent) and
// applies it as one matrix product per interaction offset:
//   * a workgroup (8 wavefronts, two per SIMD, or 4) takes a block of targets of one
//     level and child octant (they share their 189 candidate offsets); a
//     wave holds 16/nc of them, the nc components of a target side by side, as
//     the 16 columns of 16x16x32 f16 MFMA tiles;
//   * the offsets present in the block are walked grouped by azimuth: the
//     sources' columns are rotated by e^{i m phi} in FP32 registers and scaled
//     (the largest value of a column's sources to below 2^15), split as
//     x = H + L with H = f16(x), L = f16(x - H), and C += A_hi H + A_lo H +
//     A_hi L runs on the f16 matrix cores with FP32 accumulation; D_c, scaled
//     to the f16 range and split the same way, is copied into LDS by the LDS
//     DMA one offset ahead (two buffers), the sources' columns are requested one
//     offset ahead into registers;
//   * at the end of an azimuth group C is rotated back by e^{-i m phi} and
//     added into the running FP32 sum S; each target's L~ is written once in
//     FP64 at the end (the first writer of L at levels >= 2).  (Rotating the
//     accumulators from group to group instead, without S, saves registers but
//     rounds each earlier contribution once per later group: 3x the error.)
// Orders 1..12 (the class operator of order 12 fills 66 KiB).
//
// 16M Plummer p = 12: 98.2 -> 88.6 ms; 4M uniform p = 10: 27.6 -> 22.4 ms (and 2% more
// since every column has its own scale), since
//   * the columns come an offset ahead, the splits move between the products, and
//     the loop's register copies, which waited for every load in flight, are gone
//     (93.4 / 25.6);
//   * the components of a target sit in neighbouring lanes, whose loads are 64
//     contiguous bytes (one component to a wave, every lane of a load touched its
//     own line: the vector L1's accesses took 80% of the kernel's cycles).
// Of an offset's ~7,700 cycles the products take 99 x 16 x 2 per SIMD.  Left out to
// see (before the second step): the products 8%, the splits 8%, the operator copy
// 14%, its fragments' LDS reads nothing, sources always in L2 5%, operators 2%: what
// bounds it is the chain of an offset's loads, splits, products and barrier, two
// wavefronts deep on a SIMD.
#pragma once

#if !defined(__HIPCC__) && !defined(__host__)
#define __host__
#define __device__
#endif

#include <cstdint>

namespace sfmm {

constexpr int kDenseMaxP = 12;
constexpr int kDenseWaves = 8;         // most wavefronts per workgroup (two per SIMD); 4 also runs
constexpr int kDenseMaxEntries = 192;  // interaction offsets of a block (at most 189)
constexpr int kDenseMaxSlots = 32;
constexpr int kDenseMaxRows = 112;

__host__ __device__ constexpr int dceil(int a, int b) { return (a + b - 1) / b; }

// Index orders of the dense operator.
//
// Columns (K): the B operand of a 16x16x32 MFMA gives lane l the K values
// 8 (l / 16) + 0..7 of column l % 16.  Coefficients are placed in "slots" of
// four: element q of slot s sits at K = 32 (s / 8) + 8 q + s % 8, so the four
// lane groups hold the four elements of a slot in the same register, and the
// azimuth factor e^{i m phi} of a slot is one wave-uniform value when its
// elements share the order m.  Slots take the orders m >= 1, four degrees at a
// time; the orders m = 0 (no azimuth factor) fill the free places of those
// slots (their sin places stay empty), then slots of their own.  The cos and
// sin parts share the K order, so lane and register of Re c(n,m) and Im c(n,m)
// coincide and the rotation is in-lane.
// Rows: the (n, m >= 1) pairs (cos and sin rows aligned), then the cos rows of
// order 0; padded to 16-row tiles.
struct DenseOrder {
    int p = 0;
    int ns = 0;           // slots
    int nks = 0;          // 32-wide K-steps (both parts)
    int kc = 0;           // K extent of each part: 32 nks
    int npair = 0;        // (n, m >= 1) coefficients
    int mtc = 0, mts = 0; // 16-row tiles of the cos / sin part
    int kd = 0;           // floats per (node, component) in the FP32 copy: cos kc, then sin kc
    int nfrag = 0;        // 16x32 A fragments per class
    int chunks = 0;       // 1 KiB copy chunks per class (hi and lo of each fragment), padded so
                          // that every wavefront of the workgroup copies the same number
    int el[4][kDenseMaxSlots] = {};  // element (32 n + m) at (q, slot), -1 = empty
    int row[kDenseMaxRows] = {};     // element of each row, -1 = padding
};

__host__ __device__ constexpr DenseOrder dense_order(int p)
{
    DenseOrder o{};
    o.p = p;
    for (int q = 0; q < 4; ++q)
        for (int s = 0; s < kDenseMaxSlots; ++s) o.el[q][s] = -1;
    for (int r = 0; r < kDenseMaxRows; ++r) o.row[r] = -1;
    int s = 0, nr = 0;
    for (int m = 1; m <= p; ++m)
        for (int n = m; n <= p; n += 4, ++s)
            for (int q = 0; q < 4 && n + q <= p; ++q) {
                o.el[q][s] = 32 * (n + q) + m;
                o.row[nr++] = 32 * (n + q) + m;
            }
    o.npair = nr;
    // orders 0 into the free places, then slots of their own
    int n0 = 0;
    for (int t = 0; t < s && n0 <= p; ++t)
        for (int q = 0; q < 4 && n0 <= p; ++q)
            if (o.el[q][t] < 0) o.el[q][t] = 32 * n0++;
    for (; n0 <= p; ++s)
        for (int q = 0; q < 4 && n0 <= p; ++q) o.el[q][s] = 32 * n0++;
    for (int n = 0; n <= p; ++n) o.row[nr++] = 32 * n;
    o.ns = s;
    o.nks = dceil(o.ns, 8);
    o.kc = 32 * o.nks;
    o.mtc = dceil(o.npair + p + 1, 16);
    o.mts = dceil(o.npair, 16);
    o.kd = 2 * o.kc;
    o.nfrag = (o.mtc + o.mts) * o.nks;
    o.chunks = dceil(2 * o.nfrag, kDenseWaves) * kDenseWaves;
    return o;
}

// K index of element q of slot s, and back.
__host__ __device__ constexpr int dense_kidx(int s, int q) { return 32 * (s / 8) + 8 * q + s % 8; }
__host__ __device__ constexpr int dense_kslot(int k) { return 8 * (k / 32) + k % 8; }
__host__ __device__ constexpr int dense_kq(int k) { return (k % 32) / 8; }

// Element (32 n + m) at K index k of the cos (part 0) or sin (part 1) part, -1 if empty.
__host__ __device__ constexpr int dense_elem(const DenseOrder& o, int part, int k)
{
    const int s = dense_kslot(k);
    if (k < 0 || k >= o.kc || s >= o.ns) return -1;
    const int e = o.el[dense_kq(k)][s];
    return (part == 1 && e % 32 == 0) ? -1 : e;
}
// Element of row r of a part, -1 for padding.
__host__ __device__ constexpr int dense_row_elem(const DenseOrder& o, int part, int r)
{
    if (r < 0 || r >= kDenseMaxRows) return -1;
    if (part == 1 && r >= o.npair) return -1;
    return o.row[r];
}

// Real-form index (degree n at [n^2, (n+1)^2): Re c(n,0), Re c(n,1), Im c(n,1),
// ...) of element e in part `part`.
__host__ __device__ constexpr int dense_rf(int e, int part)
{
    const int n = e / 32, m = e % 32;
    if (part == 1) return n * n + 2 * m;
    return m == 0 ? n * n : n * n + 2 * m - 1;
}

// Position in the FP32 copy ([cos kc][sin kc] per node and component) of the
// real-form coefficient r.
__host__ __device__ constexpr int dense_pos(const DenseOrder& o, int r)
{
    int n = 0;
    while ((n + 1) * (n + 1) <= r) ++n;
    const int qq = r - n * n;
    const int m = (qq + 1) / 2;
    const bool sin_part = qq > 0 && qq % 2 == 0;
    const int want = 32 * n + m;
    for (int s = 0; s < o.ns; ++s)
        for (int q = 0; q < 4; ++q)
            if (o.el[q][s] == want) return (sin_part ? o.kc : 0) + dense_kidx(s, q);
    return -1;
}

// The order shared by the elements of order m >= 1 of slot s (0 if it holds
// none), and the lane groups q whose element there is of order 0 (bit q):
// their azimuth factor is 1.
__host__ __device__ constexpr int dense_slot_m(const DenseOrder& o, int s)
{
    for (int q = 0; q < 4; ++q)
        if (s < o.ns && o.el[q][s] >= 0 && o.el[q][s] % 32 != 0) return o.el[q][s] % 32;
    return 0;
}
__host__ __device__ constexpr int dense_slot_zero(const DenseOrder& o, int s)
{
    int b = 0;
    for (int q = 0; q < 4; ++q)
        if (s < o.ns && o.el[q][s] >= 0 && o.el[q][s] % 32 == 0) b |= 1 << q;
    return b;
}

// Layout of the FP32 copy of the multipoles that the mixed-precision M2L reads:
// per component `row` floats, the real-form coefficient r at place pos[r] (dense
// order for p <= 12, unpermuted above); for p <= 12 the components of a node
// alternate every four places ([node][place / 4][component][4]), so that the
// lanes of one target, its components, load 64 contiguous bytes (4 components).
template <int P>
struct F32Layout {
    static constexpr bool dense = P <= kDenseMaxP;
    static constexpr int row = dense ? dense_order(P).kd : (P + 1) * (P + 1);
    int pos[(P + 1) * (P + 1)] = {};
    constexpr F32Layout()
    {
        const DenseOrder o = dense_order(dense ? P : 1);
        for (int r = 0; r < (P + 1) * (P + 1); ++r) pos[r] = dense ? dense_pos(o, r) : r;
    }
};

template <int P>
struct F32LayoutOf {
    static constexpr F32Layout<P> L{};
};

// Azimuth groups: interaction offsets (di, dj, dk) sharing the direction of
// (di, dj) (so the same e^{i m phi}); (0, 0) joins the group of (1, 0).
constexpr int kAzGroups = 32;

}  // namespace sfmm

// ------------------------------------------------------------------ device code
#if defined(__HIPCC__)
#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.hpp"

namespace sfmm {

typedef _Float16 dh8 __attribute__((ext_vector_type(8)));
typedef float df4 __attribute__((ext_vector_type(4)));
typedef float df8 __attribute__((ext_vector_type(8)));

template <int I, int N, class F>
__device__ __forceinline__ void dense_for(F&& f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        dense_for<I + 1, N>(f);
    }
}

// x = hi + lo in f16 to 22 bits (for |x| >= 2^-3; below, to 2^-25 absolute).
// neg1 = -1 held where the compiler cannot see it: lo = f16(hi * neg1 + x) then
// stays one mixed-precision FMA (f16 operand, f32 operand, f16 result) instead
// of a conversion, a subtraction and a conversion.
__device__ __forceinline__ void dense_split(float x, _Float16& hi, _Float16& lo, float neg1)
{
    hi = static_cast<_Float16>(x);
    lo = static_cast<_Float16>(__builtin_fmaf(static_cast<float>(hi), neg1, x));
}
// -1.0f in a scalar register, opaque to constant folding.
__device__ __forceinline__ float dense_neg1()
{
    float v;
    asm volatile("s_mov_b32 %0, -1.0" : "=s"(v));
    return v;
}

// C += A_hi B_hi + A_lo B_hi + A_hi B_lo (f16 MFMA, FP32 accumulation; the
// small products first).
__device__ __forceinline__ void dense_mma(const dh8& ahi, const dh8& alo, const dh8& bhi, const dh8& blo, df4& c)
{
    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, blo, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo, bhi, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, bhi, c, 0, 0, 0);
}

// Two tiles' products, alternating: each chain of three keeps its order.
__device__ __forceinline__ void dense_mma2(const dh8* ahi, const dh8* alo, const dh8& bhi0, const dh8& blo0,
                                           const dh8& bhi1, const dh8& blo1, df4& c0, df4& c1)
{
    c0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi[0], blo0, c0, 0, 0, 0);
    c1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi[1], blo1, c1, 0, 0, 0);
    c0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo[0], bhi0, c0, 0, 0, 0);
    c1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo[1], bhi1, c1, 0, 0, 0);
    c0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi[0], bhi0, c0, 0, 0, 0);
    c1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi[1], bhi1, c1, 0, 0, 0);
}

// One 16-byte chunk per lane from global memory into LDS at dst + 16 * lane
// (LDS DMA; dst is wave-uniform).
__device__ __forceinline__ void dense_lds_copy(const dh8* src, dh8* dst)
{
    __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
}
// Keeps the compiler from moving memory operations across this point.
__device__ __forceinline__ void dense_fence() { asm volatile("" ::: "memory"); }
// Waits for every load of the wave, from memory (LDS DMA included) and from LDS.
// The builtin, not assembly: the compiler then knows that they have arrived and
// adds no wait of its own for them.
__device__ __forceinline__ void dense_wait_all()
{
    dense_fence();
    __builtin_amdgcn_s_waitcnt(7 << 4);  // vmcnt 0, lgkmcnt 0
    dense_fence();
}
// Fragment of tile t (cos tiles, then sin tiles) in K-step ks.
template <int NKS>
__host__ __device__ constexpr int ks0_frag(int t, int ks) { return t * NKS + ks; }

// The order of P as a static member (usable in constant expressions inside the
// kernel's lambdas without capturing a local).
template <int P>
struct DenseCfg {
    static constexpr DenseOrder O = dense_order(P);
};

// Adds the accumulators of one azimuth group, rotated back by e^{-i m phi}
// ((c, s) = az[2 m], az[2 m + 1]; rowm: the order of each row), into the
// running sums and clears them: (sc + i ss) += (lc + i ls) e^{-i m phi}.
// Lane group q holds rows 16 mt + 4 q + 0..3 of each tile.
template <int MTC, int MTS>
__device__ __forceinline__ void dense_flush(df4* cc, df4* cs, df4* sumc, df4* sums, const float* az,
                                            const int8_t* rowm, int q)
{
    dense_for<0, MTC>([&](auto mc) {
        constexpr int mt = decltype(mc)::value;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float lc = cc[mt][r];
            if constexpr (mt < MTS) {
                const int m = rowm[16 * mt + 4 * q + r];
                const float c = az[2 * m], sn = az[2 * m + 1], ls = cs[mt][r];
                sumc[mt][r] += __builtin_fmaf(lc, c, ls * sn);
                sums[mt][r] += __builtin_fmaf(ls, c, -(lc * sn));
            } else {
                sumc[mt][r] += lc;  // rows of order 0 (and padding)
            }
        }
        cc[mt] = df4{};
        if constexpr (mt < MTS) cs[mt] = df4{};
    });
}

template <int P, int NC, int NW>
__global__ __launch_bounds__(64 * NW, 2) void m2l_dense_kernel(DenseArgs a, const float* __restrict__ M32,
                                                           double* __restrict__ L)
{
    using Cfg = DenseCfg<P>;
    constexpr int K = (P + 1) * (P + 1);
    constexpr int TW = 16 / NC;            // targets per wave
    constexpr int TB = NW * TW;            // targets per block
    constexpr int CH = Cfg::O.chunks;      // LDS copy chunks of one class (64 x 16 bytes each)
    constexpr int NKS = Cfg::O.nks, MTC = Cfg::O.mtc, MTS = Cfg::O.mts, KC = Cfg::O.kc, KD = Cfg::O.kd;
    static_assert(MTS <= MTC && 16 * MTC <= kDenseMaxRows, "row tiles");
    static_assert(CH % NW == 0, "copy chunks per wavefront");
    // the operator of the current entry and of the next one, each [frag][hi 64 | lo 64],
    // the azimuth factors, the block's entry descriptors, and per row its order
    // and real-form indices (cos, sin)
    __shared__ dh8 opbuf0[CH * 64];
    __shared__ dh8 opbuf1[CH * 64];
    __shared__ float saz[kAzGroups * (P + 1) * 2];
    __shared__ int32_t smeta[kDenseMaxEntries];
    __shared__ int8_t srow_m[16 * MTC];
    __shared__ int16_t srow_rf[2][16 * MTC];

    const int64_t per = (a.n_block + 7) / 8;
    const int64_t blk = static_cast<int64_t>(blockIdx.x % 8) * per + blockIdx.x / 8;
    if (blk >= a.n_block) return;
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // scalar: so are the copy's and the buffers' offsets
    const int col = lane & 15, comp = col - (col / NC) * NC;
    const bool used = col / NC < TW;  // 3 components: the last column is empty
    const int ti = w * TW + (used ? col / NC : 0);
    const int32_t tg = used ? a.blk_tgt[blk * TB + ti] : -1;
    const int64_t e0 = a.blk_row[blk];
    const int ne = static_cast<int>(a.blk_row[blk + 1] - e0);

    // scale of this lane's column (one component of one target): the largest
    // |value| over its sources maps below 2^15, so rotated values stay below
    // 2^15.5 < 65504 and keep 22 bits down to 2^-18 of the largest.  A scale shared
    // by several components would take those bits from the smaller ones, which
    // differ by any factor (the caller's charges; potential and gradient by the
    // length unit).  The four lanes of a column take the same
    float mx = 0.0f;
    if (tg >= 0 && q == 0) {
        for (int i0 = 0; i0 < ne; i0 += 8) {
            int32_t sn[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) sn[u] = i0 + u < ne ? a.ent_src[(e0 + i0 + u) * TB + ti] : -1;
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (sn[u] >= 0) mx = fmaxf(mx, a.nodemax[static_cast<int64_t>(sn[u]) * NC + comp]);
        }
    }
    for (int o = 32; o > 8; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    int sexp = 0;
    if (mx > 0.0f) {
        int ex;
        (void)frexpf(mx, &ex);  // mx < 2^ex
        sexp = min(15 - ex, 127);  // a finite scale also for the smallest FP32 values
    }
    const float sc = ldexpf(1.0f, sexp);
    const float neg1 = dense_neg1();
    // a wave-uniform float held in a scalar register
    auto uniform = [](float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); };

    // copies this wavefront's CH / NW chunks of 1 KiB of the operator of class cls into
    // an LDS buffer
    auto dma = [&](int cls, dh8* __restrict__ buf, int lane) {
        const dh8* src = static_cast<const dh8*>(a.ops) + static_cast<int64_t>(cls) * CH * 64;
#pragma unroll
        for (int c = 0; c < CH / NW; ++c)
            dense_lds_copy(src + (w + NW * c) * 64 + lane, buf + (w + NW * c) * 64);
    };
    auto src_ptr = [&](int32_t s) -> const float* {
        const float* real = M32 + static_cast<int64_t>(s < 0 ? 0 : s) * NC * KD + 4 * comp;
        return (used && s >= 0) ? real : a.zero;
    };
    for (int k = tid; k < kAzGroups * (P + 1) * 2; k += 64 * NW) saz[k] = a.az[k];
    for (int k = tid; k < ne; k += 64 * NW) smeta[k] = a.ent_meta[e0 + k];
    for (int k = tid; k < 16 * MTC; k += 64 * NW) {
        const int ec = dense_row_elem(Cfg::O, 0, k), es = dense_row_elem(Cfg::O, 1, k);
        srow_m[k] = static_cast<int8_t>(ec < 0 ? 0 : ec % 32);
        srow_rf[0][k] = static_cast<int16_t>(ec < 0 ? -1 : dense_rf(ec, 0));
        srow_rf[1][k] = static_cast<int16_t>(es < 0 ? -1 : dense_rf(es, 1));
    }

    // accumulators of the current azimuth group, and the running sums (unrotated frame)
    df4 cc[MTC], cs[MTS], sumc[MTC], sums[MTS];
    for (int i = 0; i < MTC; ++i) cc[i] = sumc[i] = df4{};
    for (int i = 0; i < MTS; ++i) cs[i] = sums[i] = df4{};
    // the source columns of every K-step (lane group q holds K = 8 q + 0..7 of each
    // 32-wide K-step, cos and sin), requested one entry ahead: a K-step's
    // registers take the next entry's columns as soon as they are split.  (One
    // K-step ahead, the columns queued behind the operator copy.)
    df8 xr[NKS], xi[NKS];
    for (int ks = 0; ks < NKS; ++ks) xr[ks] = xi[ks] = df8{};
    auto load_step = [&](const float* p, auto kc, int q) {
        constexpr int ks = decltype(kc)::value;
        // places 32 ks + 8 q + 0..7, in two pieces of four, NC components apart
        const df4* c = reinterpret_cast<const df4*>(p) + (8 * ks + 2 * q) * NC;
        const df4* d = c + KC / 4 * NC;
        xr[ks] = __builtin_shufflevector(c[0], c[NC], 0, 1, 2, 3, 4, 5, 6, 7);
        xi[ks] = __builtin_shufflevector(d[0], d[NC], 0, 1, 2, 3, 4, 5, 6, 7);
    };
    int32_t src1 = -1;  // this lane's source of the next entry
    if (ne > 0) {
        dma(a.ent_meta[e0] & 0xff, opbuf0, lane);
        const float* csp = src_ptr(a.ent_src[e0 * TB + ti]);
        src1 = a.ent_src[(e0 + (ne > 1 ? 1 : 0)) * TB + ti];
        if (ne < 2) src1 = -1;
        dense_for<0, NKS>([&](auto kc) {
            load_step(csp, kc, q);
        });
    }
    __syncthreads();  // saz, smeta, srow_*
    float csx[P + 1], csy[P + 1];  // cos, sin of m phi of the current azimuth group
    auto factors = [&](int g) {
        for (int m = 0; m <= P; ++m) {
            csx[m] = uniform(saz[(g * (P + 1) + m) * 2]);
            csy[m] = uniform(saz[(g * (P + 1) + m) * 2 + 1]);
        }
    };
    int i = 0, g = -1;
    if (ne > 0) {
        g = __builtin_amdgcn_readfirstlane((smeta[0] >> 8) & 0xff);
        factors(g);
    }
    // one entry, returning the group of the next (-1: none); even entries read opbuf0
    // and fill opbuf1, odd ones the reverse (two arrays, so the reads are seen not to
    // alias the copy in flight)
    auto entry = [&](const dh8* __restrict__ cur, dh8* __restrict__ nxt) {
        const bool more = i + 1 < ne;
        // the lane and its group, re-read each entry, so that the addresses and the
        // per-lane azimuth factors of the slots shared by orders m and 0 are formed
        // where they are used instead of being held in registers across the loop
        // (which spilled the running sums)
        int qv = q, lv = lane;
        asm volatile("" : "+v"(qv), "+v"(lv));
        const int nmeta = __builtin_amdgcn_readfirstlane(smeta[more ? i + 1 : i]);
        // the operator of entry i is in LDS, this entry's columns are in registers
        // (requested during the previous entry), and every wave is done with entry
        // i - 1.  One wait for all of it before the next copy is issued: behind a copy
        // in flight the compiler waits for everything, the copy included
        dense_wait_all();
        __builtin_amdgcn_s_barrier();
        dense_fence();
        // The next operator's copy is issued whole (the wavefronts queue for it before
        // their first products, 1,700 cycles of an entry's 8,500; spread between the
        // K-steps it was slower).  After the last entry once more, unused: a branch
        // would make the compiler wait for every load in flight.
        const int ncls = nmeta & 0xff;
        dma(ncls, nxt, lv);
        dense_fence();
        const float* nsp = src_ptr(src1);
        asm volatile("" ::"v"(nsp));  // src1 is used up before its register is loaded again
        src1 = a.ent_src[(e0 + (i + 2 < ne ? i + 2 : ne - 1)) * TB + ti];
        {
            // A fragments of the 11-ish tiles of each K-step, in pairs of tiles whose
            // chains of three products alternate, one pair ahead (the fences keep the
            // compiler from loading further ahead, which would take the registers of
            // the accumulators); tile t of K-step ks is fragment t * NKS + ks (cos
            // tiles, then sin tiles)
            constexpr int NT = MTC + MTS, NTP = (NT + 1) / 2;
            dh8 ah[2], al[2];
            auto fetch = [&](auto pc, auto kc, dh8* h, dh8* l) {
                constexpr int t = 2 * decltype(pc)::value, ks = decltype(kc)::value;
                h[0] = cur[ks0_frag<NKS>(t, ks) * 128 + lv];
                l[0] = cur[ks0_frag<NKS>(t, ks) * 128 + 64 + lv];
                if constexpr (t + 1 < NT) {
                    h[1] = cur[ks0_frag<NKS>(t + 1, ks) * 128 + lv];
                    l[1] = cur[ks0_frag<NKS>(t + 1, ks) * 128 + 64 + lv];
                }
            };
            fetch(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, ah, al);
            // B fragments of a K-step: the columns scaled, rotated by e^{i m phi} and split,
            // slot by slot (the fused products written out, here and in the flush: which
            // of two products is fused would otherwise change with the code around).
            // Those of K-step ks + 1 are made between the products of K-step ks (two
            // sets), in the shadow of the matrix cores; before, all wavefronts split and
            // then all multiplied.
            dh8 bch[2], bcl[2], bsh[2], bsl[2];
            auto split = [&](auto kc, auto jc) {
                constexpr int ks = decltype(kc)::value, j = decltype(jc)::value, B = ks & 1;
                constexpr int s = 8 * ks + j;
                constexpr int m = dense_slot_m(Cfg::O, s), z = dense_slot_zero(Cfg::O, s);
                float cm = csx[m], sm = csy[m];
                if constexpr (z != 0 && m != 0) {  // lane groups whose element is of order 0
                    const bool zq = (z >> qv) & 1;
                    cm = zq ? 1.0f : cm;
                    sm = zq ? 0.0f : sm;
                }
                // the scale, a power of two: exact.  (On the columns, 16 multiplies per
                // K-step and 1.4-1.8% of the evaluation: 4M uniform p = 10 29.6 -> 30.1 ms,
                // 16M Plummer p = 12 120.8 -> 122.5.  One scale per wavefront would go into
                // the azimuth factors.)
                const float xrj = xr[ks][j] * sc, xij = xi[ks][j] * sc;
                _Float16 hh, ll;
                dense_split(__builtin_fmaf(xrj, cm, -(xij * sm)), hh, ll, neg1);
                bch[B][j] = hh;
                bcl[B][j] = ll;
                dense_split(__builtin_fmaf(xij, cm, xrj * sm), hh, ll, neg1);
                bsh[B][j] = hh;
                bsl[B][j] = ll;
            };
            dense_for<0, 8>([&](auto jc) { split(std::integral_constant<int, 0>{}, jc); });
            dense_for<0, NKS>([&](auto kc) {
                constexpr int ks = decltype(kc)::value;
                __builtin_amdgcn_sched_barrier(0);
                // the next entry's columns of this K-step, whose columns are split
                // already (zeros after the last entry)
                load_step(nsp, kc, qv);
                dense_for<0, NTP>([&](auto pc) {
                    constexpr int pr = decltype(pc)::value, t = 2 * pr;
                    constexpr int pn = (pr + 1) % NTP, kn = pr + 1 < NTP ? ks : ks + 1;
                    dh8 nh[2], nl[2];
                    dense_fence();
                    if constexpr (kn < NKS)
                        fetch(std::integral_constant<int, pn>{}, std::integral_constant<int, kn>{}, nh, nl);
                    df4& c0 = t < MTC ? cc[t < MTC ? t : 0] : cs[t < MTC ? 0 : t - MTC];
                    constexpr int B = ks & 1;
                    const dh8& h0 = t < MTC ? bch[B] : bsh[B];
                    const dh8& l0 = t < MTC ? bcl[B] : bsl[B];
                    if constexpr (t + 1 < NT) {
                        constexpr int u = t + 1;
                        df4& c1 = u < MTC ? cc[u < MTC ? u : 0] : cs[u < MTC ? 0 : u - MTC];
                        dense_mma2(ah, al, h0, l0, u < MTC ? bch[B] : bsh[B], u < MTC ? bcl[B] : bsl[B], c0, c1);
                    } else {
                        dense_mma(ah[0], al[0], h0, l0, c0);
                    }
                    if constexpr (ks + 1 < NKS)
                        dense_for<8 * pr / NTP, 8 * (pr + 1) / NTP>(
                            [&](auto jc) { split(std::integral_constant<int, ks + 1>{}, jc); });
                    if constexpr (kn < NKS) {
                        ah[0] = nh[0], al[0] = nl[0];
                        if constexpr (2 * pn + 1 < NT) ah[1] = nh[1], al[1] = nl[1];
                    }
                });
            });
        }
        return more ? (nmeta >> 8) & 0xff : -1;
    };
    // after an entry: at the end of its group, the contribution, rotated back, into
    // the running sums.  Even and odd entries follow each other in the text: a
    // choice between two calls merges their registers by copies, which wait for the
    // loads in flight (700-1100 cycles an entry)
    auto next_group = [&](int gn) {
        ++i;
        if (gn == g) return;
        dense_flush<MTC, MTS>(cc, cs, sumc, sums, saz + g * (P + 1) * 2, srow_m, q);
        g = gn;
        if (g >= 0) factors(g);
    };
    while (g >= 0) {
        next_group(entry(opbuf0, opbuf1));
        if (g < 0) break;
        next_group(entry(opbuf1, opbuf0));
    }
    dense_wait_all();  // no copy into LDS outlives the workgroup
    // L~ of the block's targets (first writer at its level), unscaled, in FP64
    if (tg < 0) return;
    const double un = ldexp(1.0, -a.op_exp - sexp);
    double* Lt = L + (static_cast<int64_t>(tg) * NC + comp) * K;
    dense_for<0, MTC>([&](auto mc) {
        constexpr int mt = decltype(mc)::value;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * mt + 4 * q + r;
            const int rc = srow_rf[0][row];
            if (rc >= 0) Lt[rc] = static_cast<double>(sumc[mt][r]) * un;
            if constexpr (mt < MTS) {
                const int rs = srow_rf[1][row];
                if (rs >= 0) Lt[rs] = static_cast<double>(sums[mt][r]) * un;
            }
        }
    });
}

template <int P, int NW>
void launch_m2l_dense_pw(const DenseArgs& a, int nc, const float* M32, double* L, hipStream_t s)
{
    const dim3 grid(static_cast<unsigned>(8 * ((a.n_block + 7) / 8))), blk(64 * NW);
    switch (nc) {
    case 1: hipLaunchKernelGGL((m2l_dense_kernel<P, 1, NW>), grid, blk, 0, s, a, M32, L); break;
    case 2: hipLaunchKernelGGL((m2l_dense_kernel<P, 2, NW>), grid, blk, 0, s, a, M32, L); break;
    case 3: hipLaunchKernelGGL((m2l_dense_kernel<P, 3, NW>), grid, blk, 0, s, a, M32, L); break;
    default: hipLaunchKernelGGL((m2l_dense_kernel<P, 4, NW>), grid, blk, 0, s, a, M32, L); break;
    }
}

// a.waves (4 or 8) wavefronts per workgroup: the tile shape, which fixes the
// targets per block the work lists were cut for (16/nc per wavefront).
template <int P>
void launch_m2l_dense_p(const DenseArgs& a, int nc, const float* M32, double* L, hipStream_t s)
{
    if (a.waves == 4) launch_m2l_dense_pw<P, 4>(a, nc, M32, L, s);
    else launch_m2l_dense_pw<P, 8>(a, nc, M32, L, s);
}

}  // namespace sfmm
#endif
