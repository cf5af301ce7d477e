// Device side of the broadcast M2L (m2l_bcast.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "m2l_bcast.hpp"

namespace sfmm {

namespace {

namespace bc {

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

template <int W, int NW, class F>
__device__ __forceinline__ void for_wave(int w, F&& f)
{
    if constexpr (W < NW) {
        if (w == W) f(std::integral_constant<int, W>{});
        else for_wave<W + 1, NW>(w, f);
    }
}

__host__ __device__ constexpr int rc(int n, int m) { return m == 0 ? n * n : n * n + 2 * m - 1; }
__host__ __device__ constexpr int rs(int n, int m) { return n * n + 2 * m; }
// X row of coefficient (n, m, part)
__host__ __device__ constexpr int row_of(int mode, int n, int m, int part)
{
    return mode == kBcastBoth ? (part == 0 ? rc(n, m) : rs(n, m))
                              : (part == 0 ? n * (n + 1) / 2 + m : n * (n - 1) / 2 + m - 1);
}

// c += op[lane LN of this lane's 16-lane row] * x.  The compiler does not form
// this instruction from v_mov_b64_dpp and v_fma_f64, hence the asm.  A DPP read
// needs two wait states after a vector write of op: op comes from memory, an s_nop
// separates it from the copies at a change of class, and a test follows every path
// through the built kernels back from the reads for any copy of the compiler's.  (An
// s_nop in every step took 0.6% of the M2L: 16M Plummer p = 12 177.8 -> 179.0 ms.)
template <int LN>
__device__ __forceinline__ void fmac_row(double& c, double op, double x)
{
    asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(c) : "v"(op), "v"(x), "n"(LN));
}
template <int LN>
__device__ __forceinline__ void fnmac_row(double& c, double op, double x)
{
    asm("v_fmac_f64_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(c) : "v"(op), "v"(x), "n"(LN));
}

struct alignas(16) D2 {
    double x, y;
};

template <int N>
struct Regs {
    double v[N > 0 ? N : 1];
};

// Loads of N operator registers: lane l gets element 16 r + l % 16.
template <int N>
__device__ __forceinline__ void load_ops(double* r, const double* p, int lane)
{
#pragma unroll
    for (int k = 0; k < N; ++k) r[k] = p[k * 16 + (lane & 15)];
}

__device__ __forceinline__ void barrier_lds()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int P, bool COAX, int MODE>
inline constexpr BcastUnits kUnits = bcast_units(P, COAX, MODE);

// A stage's work of one wavefront as a list of operator columns (block q, column b).
struct ColumnList {
    int n = 0;
    int q[320] = {};
    int b[320] = {};
};
template <int P, bool COAX, int MODE, int W>
constexpr ColumnList column_list()
{
    ColumnList c;
    const BcastUnits& u = kUnits<P, COAX, MODE>;
    for (int q = 0; q < u.count[W]; ++q)
        for (int b = 0; b < bcast_size(P, COAX, u.idx[W][q], u.part[W][q]); ++b) {
            c.q[c.n] = q;
            c.b[c.n] = b;
            ++c.n;
        }
    return c;
}

template <int P, int NC, int MODE, int W>
struct Wave {
    static constexpr int NW = bcast_waves(P);
    // columns read from LDS ahead of their use (fewer where registers are short)
    static constexpr int kAheadX = P >= 16 ? 3 : 6;
    static constexpr const BcastUnits& UR = kUnits<P, false, MODE>;
    static constexpr const BcastUnits& UT = kUnits<P, true, MODE>;
    static constexpr int NR = bcast_regs(P, UR, false, W), NT = bcast_regs(P, UT, true, W);
    static constexpr int NB = NR > NT ? NR : NT;
    static constexpr int RR = bcast_reg0(P, UR, false, NW), RT = bcast_reg0(P, UT, true, NW);
    static constexpr int R0 = bcast_reg0(P, UR, false, W), T0 = bcast_reg0(P, UT, true, W);
    static constexpr int NU = UR.count[W], NV = UT.count[W];
    static constexpr ColumnList CR = column_list<P, false, MODE, W>(), CT = column_list<P, true, MODE, W>();
    // degrees of this wavefront: a degree whose cos and sin blocks are both here
    // appears once in the columns and accumulators
    static constexpr bool first_of(int q)
    {
        for (int k = 0; k < q; ++k)
            if (UR.idx[W][k] == UR.idx[W][q]) return false;
        return true;
    }
    // first column / accumulator pair of block q's degree
    static constexpr int col0(int q)
    {
        int o = 0;
        for (int k = 0; k < NU; ++k) {
            if (UR.idx[W][k] == UR.idx[W][q]) return o;
            if (first_of(k)) o += UR.idx[W][k] + 1;
        }
        return o;
    }
    static constexpr int ncols()
    {
        int o = 0;
        for (int k = 0; k < NU; ++k)
            if (first_of(k)) o += UR.idx[W][k] + 1;
        return o;
    }
    static constexpr int NCOL = ncols();

    Regs<NR> rot;   // rotation of the step's class: forward, and transposed the back rotation
    Regs<NB> bank;  // coaxial operator, then the next class's rotation
    D2 col[NCOL > 0 ? NCOL : 1];                                // gathered (Re, Im) of the step's columns
    double are[NCOL > 0 ? NCOL : 1], aim[NCOL > 0 ? NCOL : 1];  // accumulators

    // gathered pair j of NCOL: the pair's index in a node, and whether Im is used
    struct Pair {
        int index = 0;
        bool im = false;
    };
    static constexpr Pair pair_of(int j)
    {
        for (int q = 0; q < NU; ++q) {
            const int n = UR.idx[W][q], m = j - col0(q);
            if (first_of(q) && m >= 0 && m <= n) return Pair{bcast_pair(n, m), m > 0};
        }
        return Pair{};
    }
    template <int J>
    __device__ __forceinline__ void load_col(const D2* __restrict__ p)
    {
        constexpr Pair pr = pair_of(J);
        if constexpr (MODE == kBcastSin && !pr.im) return;  // order 0 has no sin part
        else if constexpr (pr.im) col[J] = p[pr.index * NC];
        else col[J].x = p[pr.index * NC].x;
    }
    __device__ __forceinline__ void load_cols(const D2* __restrict__ p)
    {
        static_for<0, NCOL>([&](auto jc) { load_col<decltype(jc)::value>(p); });
    }

    // 1: azimuth (cm1 = cos m phi - 1, s = sin m phi in lane m - 1 of each row) and forward rotation
    __device__ __forceinline__ void stage1(double* X, int lane, double cm1, double s) const
    {
        double y[P + 1];
        auto column = [&](auto kc) {
            constexpr int k = decltype(kc)::value, q = CR.q[k];
            constexpr int part = UR.part[W][q], m = CR.b[k] + part;
            const D2 v = col[col0(q) + m];
            double t = part == 0 ? v.x : v.y;
            if constexpr (m > 0) {
                const double own = t;
                fmac_row<m - 1>(t, cm1, own);
                if constexpr (part == 0) fnmac_row<m - 1>(t, s, v.y);
                else fmac_row<m - 1>(t, s, v.x);
            }
            return t;
        };
        double x[2];
        if constexpr (CR.n > 0) x[0] = column(std::integral_constant<int, 0>{});
        static_for<0, CR.n>([&](auto kc) {
            constexpr int k = decltype(kc)::value, q = CR.q[k], b = CR.b[k];
            constexpr int n = UR.idx[W][q], part = UR.part[W][q];
            constexpr int S = bcast_size(P, false, n, part), E = bcast_block(P, UR, false, W, q);
            if constexpr (k + 1 < CR.n) x[(k + 1) & 1] = column(std::integral_constant<int, k + 1>{});
            static_for<0, S>([&](auto ac) {
                constexpr int a = decltype(ac)::value, e = E + b * S + a;
                if constexpr (b == 0) y[a] = 0.0;
                fmac_row<e % 16>(y[a], rot.v[e / 16], x[k & 1]);
                if constexpr (b == S - 1) X[row_of(MODE, n, a + part, part) * 64 + lane] = y[a];
            });
            __builtin_amdgcn_sched_barrier(0);
        });
    }

    // The next step's columns are requested on the way through stages 2 and 3, a
    // few per operator column: requested all at once they fill the memory
    // pipeline and hold up the products behind them.
    static constexpr int LD2 = NCOL / 2;
    template <int FROM, int TO>
    __device__ __forceinline__ void load_some(const D2* __restrict__ p)
    {
        static_for<FROM, TO>([&](auto jc) { load_col<decltype(jc)::value>(p); });
    }

    // 2: coaxial translation in place
    __device__ __forceinline__ void stage2(double* X, int lane, const D2* __restrict__ p)
    {
        double y[P + 1], x[kAheadX];
        auto read = [&](auto kc) {
            constexpr int k = decltype(kc)::value, q = CT.q[k];
            constexpr int m = UT.idx[W][q], part = UT.part[W][q];
            x[k % kAheadX] = X[row_of(MODE, m + CT.b[k], m, part) * 64 + lane];
        };
        static_for<0, (CT.n < kAheadX ? CT.n : kAheadX)>(read);
        static_for<0, CT.n>([&](auto kc) {
            constexpr int k = decltype(kc)::value, q = CT.q[k], b = CT.b[k];
            constexpr int m = UT.idx[W][q], part = UT.part[W][q];
            constexpr int S = bcast_size(P, true, m, part), E = bcast_block(P, UT, true, W, q);
            static_for<0, S>([&](auto ac) {
                constexpr int a = decltype(ac)::value, e = E + b * S + a;
                if constexpr (b == 0) y[a] = 0.0;
                fmac_row<e % 16>(y[a], bank.v[e / 16], x[k % kAheadX]);
                if constexpr (b == S - 1) X[row_of(MODE, m + a, m, part) * 64 + lane] = y[a];
            });
            if constexpr (k + kAheadX < CT.n) read(std::integral_constant<int, k + kAheadX>{});
            load_some<LD2 * k / CT.n, LD2*(k + 1) / CT.n>(p);
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (CT.n == 0) load_some<0, LD2>(p);
    }

    // 3: back rotation (the forward operator transposed), azimuth e^{-i m phi}
    // (c, s in lane m - 1), accumulation
    __device__ __forceinline__ void stage3(const double* X, int lane, double c, double s, const D2* __restrict__ p)
    {
        double y[P + 1], x[kAheadX];
        auto read = [&](auto kc) {
            constexpr int k = decltype(kc)::value, q = CR.q[k];
            constexpr int n = UR.idx[W][q], part = UR.part[W][q];
            x[k % kAheadX] = X[row_of(MODE, n, CR.b[k] + part, part) * 64 + lane];
        };
        static_for<0, (CR.n < kAheadX ? CR.n : kAheadX)>(read);
        static_for<0, CR.n>([&](auto kc) {
            constexpr int k = decltype(kc)::value, q = CR.q[k], b = CR.b[k];
            constexpr int n = UR.idx[W][q], part = UR.part[W][q];
            constexpr int S = bcast_size(P, false, n, part), E = bcast_block(P, UR, false, W, q);
            static_for<0, S>([&](auto ac) {
                constexpr int a = decltype(ac)::value, e = E + a * S + b;
                if constexpr (b == 0) y[a] = 0.0;
                fmac_row<e % 16>(y[a], rot.v[e / 16], x[k % kAheadX]);
            });
            if constexpr (k + kAheadX < CR.n) read(std::integral_constant<int, k + kAheadX>{});
            constexpr int kn = CR.n * 3 / 4 > 0 ? CR.n * 3 / 4 : 1;
            if constexpr (k < kn) load_some<LD2 + (NCOL - LD2) * k / kn, LD2 + (NCOL - LD2) * (k + 1) / kn>(p);
            if constexpr (b == S - 1) {
                static_for<0, S>([&](auto ac) {
                    constexpr int a = decltype(ac)::value;
                    constexpr int m = a + part, j = col0(q) + m;
                    if constexpr (m == 0) {
                        are[j] += y[a];
                    } else if constexpr (part == 0) {
                        fmac_row<m - 1>(are[j], c, y[a]);
                        fnmac_row<m - 1>(aim[j], s, y[a]);
                    } else {
                        fmac_row<m - 1>(are[j], s, y[a]);
                        fmac_row<m - 1>(aim[j], c, y[a]);
                    }
                });
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    }
};

// The local expansion that this lane's columns belong to (null: none).
template <int P, int NC>
__device__ __forceinline__ double* lane_target(const BcastArgs& a, int64_t g, int lane, double* L)
{
    constexpr int TB = 16 / NC;
    const int l = lane & 15, t = l / NC, c = l - (l / NC) * NC;
    const int32_t tg = t < TB ? a.grp_tgt[g * (4 * TB) + (lane >> 4) * TB + t] : -1;
    return tg < 0 ? nullptr : L + (static_cast<int64_t>(tg) * NC + c) * ((P + 1) * (P + 1));
}

}  // namespace bc

// One workgroup: steps [s0, s1) of a group of four rows.  The accumulated columns
// are left in X ([coefficient][64 lanes]) or, where a kernel runs one part (a
// wavefront's accumulators are then the part's whole result), written: to the
// run's partial sums, or to the targets' L (sin: added).
template <int P, int NC, int MODE, int W>
__device__ __forceinline__ void bcast_wave(const BcastArgs& a, int64_t g, int64_t s0, int64_t s1, int64_t prow, double* X,
                                           double* __restrict__ L)
{
    using namespace bc;
    using WV = Wave<P, NC, MODE, W>;
    constexpr int TB = 16 / NC;
    constexpr int NP = bcast_pairs(P);
    const int lane = threadIdx.x & 63;
    const int row = lane >> 4, l = lane & 15;
    const int t = l / NC < TB ? l / NC : TB - 1;
    const int comp = l / NC < TB ? l - (l / NC) * NC : NC - 1;  // a spare lane repeats the last column
    const int az_l = l < P ? l : P - 1;
    WV wv;
#pragma unroll
    for (int k = 0; k < (WV::NCOL > 0 ? WV::NCOL : 1); ++k) wv.are[k] = wv.aim[k] = 0.0;

    const D2* Mx = reinterpret_cast<const D2*>(a.Mx) + comp;
    // steps are counted from s0 in 32 bits
    const int ns = static_cast<int>(s1 - s0);
    const int32_t* srcs = a.step_src + s0 * (4 * TB) + row * TB + t;
    const int32_t* words = a.step_meta + s0 * 4 + row;
    auto cols = [&](int32_t src) { return Mx + static_cast<int64_t>(src) * (NP * NC); };
    auto cls_of = [](int w) { return __builtin_amdgcn_readfirstlane((w >> 9) & 127); };
    auto d2_of = [](int w) { return __builtin_amdgcn_readfirstlane(w >> 16); };
    auto az = [&](int w) { return (w & 511) * 16 + az_l; };
    auto rot_ops = [&](int w) { return a.rot + (static_cast<int64_t>(cls_of(w)) * WV::RR + WV::R0) * 16; };
    auto cox_ops = [&](int w) { return a.coax + (static_cast<int64_t>(d2_of(w)) * WV::RT + WV::T0) * 16; };
    const D2* azf = reinterpret_cast<const D2*>(a.az_fwd);
    const D2* azb = reinterpret_cast<const D2*>(a.az_back);

    if (ns > 0) {
        int w = words[0];
        load_ops<WV::NR>(wv.rot.v, rot_ops(w), lane);
        wv.load_cols(cols(srcs[0]));
        D2 f = azf[az(w)], b = azb[az(w)];
        const int n1 = ns > 1 ? 1 : 0;
        int32_t src_n = srcs[n1 * (4 * TB)];
        int wn = words[n1 * 4];
        bool change = true;  // the class of this step is not that of the one before it
        for (int st = 0; st < ns; ++st) {
            // the columns have arrived before the coaxial operator is asked for,
            // so that no wait for a column also waits for it
            asm volatile("" : "+v"(wv.col[WV::NCOL > 0 ? WV::NCOL - 1 : 0].x), "+v"(src_n), "+v"(wn), "+v"(f.x), "+v"(b.x));
            if (change) {
#pragma unroll
                for (int k = 0; k < WV::NR; ++k)
                    if (st > 0) wv.rot.v[k] = wv.bank.v[k];
                load_ops<WV::NT>(wv.bank.v, cox_ops(w), lane);
                asm volatile("s_nop 1");
            }
            __builtin_amdgcn_sched_barrier(0);
            change = cls_of(wn) != cls_of(w);
            wv.stage1(X, lane, f.x, f.y);
            barrier_lds();
            // the next step's azimuth and columns, and the words of the one after it
            const D2* next = cols(src_n);
            f = azf[az(wn)];
            const D2 bn = azb[az(wn)];
            const int nn = st + 2 < ns ? st + 2 : ns - 1;
            src_n = srcs[nn * (4 * TB)];
            const int wnn = words[nn * 4];
            __builtin_amdgcn_sched_barrier(0);
            wv.stage2(X, lane, next);
            if (change) load_ops<WV::NR>(wv.bank.v, rot_ops(wn), lane);
            barrier_lds();
            wv.stage3(X, lane, b.x, b.y, next);
            b = bn;
            w = wn;
            wn = wnn;
        }
    }
    if constexpr (MODE != kBcastBoth) {
        double* part = prow < 0 ? nullptr : a.partial + prow * ((P + 1) * (P + 1) * 64);
        double* Lt = lane_target<P, NC>(a, g, lane, L);
        static_for<0, WV::NU>([&](auto qc) {
            constexpr int n = WV::UR.idx[W][decltype(qc)::value];
            static_for<(MODE == kBcastSin ? 1 : 0), n + 1>([&](auto mc) {
                constexpr int m = decltype(mc)::value;
                constexpr int k = WV::col0(decltype(qc)::value) + m;
                const double re = m == 0 ? wv.are[k] * 1.4142135623730951 : wv.are[k];
                if (part) {
                    part[rc(n, m) * 64 + lane] = re;
                    if constexpr (m > 0) part[rs(n, m) * 64 + lane] = wv.aim[k];
                } else if (Lt) {
                    Lt[rc(n, m)] = MODE == kBcastSin ? Lt[rc(n, m)] + re : re;
                    if constexpr (m > 0) Lt[rs(n, m)] = MODE == kBcastSin ? Lt[rs(n, m)] + wv.aim[k] : wv.aim[k];
                }
            });
            if constexpr (MODE == kBcastSin)
                if (part) part[rc(n, 0) * 64 + lane] = 0.0;
        });
        if constexpr (MODE == kBcastSin && W == 0)
            if (part) part[lane] = 0.0;  // degree 0
        return;
    } else {
    // accumulators to X rows, order 0 back in the plan's scale: a degree split
    // over two wavefronts adds in two turns
    static_for<0, 2>([&](auto turn) {
        barrier_lds();
        static_for<0, WV::NU>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            constexpr int n = WV::UR.idx[W][q], part = WV::UR.part[W][q];
            constexpr bool both = WV::UR.has(W, n, 1 - part) || n == 0;
            if constexpr (WV::first_of(q) && (decltype(turn)::value == 0) == (both || part == 0)) {
                static_for<0, n + 1>([&](auto mc) {
                    constexpr int m = decltype(mc)::value;
                    constexpr int k = WV::col0(q) + m;
                    double* xr = X + rc(n, m) * 64 + lane;
                    double* xi = X + rs(n, m) * 64 + lane;
                    if constexpr (decltype(turn)::value == 0) {
                        *xr = m == 0 ? wv.are[k] * 1.4142135623730951 : wv.are[k];
                        if constexpr (m > 0) *xi = wv.aim[k];
                    } else if constexpr (m > 0) {
                        *xr += wv.are[k];
                        *xi += wv.aim[k];
                    }
                });
            }
        });
    });
    barrier_lds();
    }
}

// L (or, when the group's steps are cut into several runs, the run's partial
// sums) written once per target.
template <int P, int NC, int MODE>
__global__ __launch_bounds__(64 * bcast_waves(P), bcast_simd_waves(P)) void m2l_bcast_kernel(BcastArgs a,
                                                                                            double* __restrict__ L)
{
    constexpr int NW = bcast_waves(P), NTH = 64 * NW;
    constexpr int K = (P + 1) * (P + 1);
    __shared__ double X[bcast_rows(P, MODE) * 64];
    const int64_t* item = a.item + 4 * static_cast<int64_t>(blockIdx.x);
    const int64_t g = item[0], s0 = item[1], s1 = item[2], prow = item[3];
    if (g < 0) return;
    bc::for_wave<0, NW>(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6), [&](auto wc) {
        bcast_wave<P, NC, MODE, decltype(wc)::value>(a, g, s0, s1, prow, X, L);
    });
    if constexpr (MODE == kBcastBoth) {
        if (prow >= 0) {
            double* part = a.partial + prow * (K * 64);
            for (int i = threadIdx.x; i < K * 64; i += NTH) part[i] = X[i];
        } else if (double* Lt = bc::lane_target<P, NC>(a, g, threadIdx.x & 63, L)) {
            for (int r = threadIdx.x >> 6; r < K; r += NW) Lt[r] = X[r * 64 + (threadIdx.x & 63)];
        }
    }
}

// L from the partial sums of a group's runs, added in run order.
template <int P, int NC>
__global__ __launch_bounds__(256) void m2l_bcast_reduce_kernel(BcastArgs a, double* __restrict__ L)
{
    constexpr int K = (P + 1) * (P + 1);
    constexpr int TB = 16 / NC;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int64_t q = i / (K * 64);
    if (q >= a.n_split) return;
    const int k = static_cast<int>(i - q * (K * 64));
    const int r = k >> 6, lane = k & 63;
    const int l = lane & 15, t = l / NC, c = l - (l / NC) * NC;
    if (t >= TB) return;
    const int32_t tg = a.grp_tgt[a.split[3 * q] * (4 * TB) + (lane >> 4) * TB + t];
    if (tg < 0) return;
    const double* p = a.partial + a.split[3 * q + 1] * (K * 64) + k;
    const int n = static_cast<int>(a.split[3 * q + 2]);
    double v = 0.0;
    for (int run = 0; run < n; ++run) v += p[static_cast<int64_t>(run) * (K * 64)];
    if constexpr (bcast_parted(P)) {
        p += a.n_partial * (K * 64);
        for (int run = 0; run < n; ++run) v += p[static_cast<int64_t>(run) * (K * 64)];
    }
    L[(static_cast<int64_t>(tg) * NC + c) * K + r] = v;
}

template <int P, int NC>
void bcast_launch(const BcastArgs& a, double* L, hipStream_t s)
{
    const dim3 grid(static_cast<unsigned>(a.n_item)), blk(64 * bcast_waves(P));
    if constexpr (bcast_parted(P)) {
        hipLaunchKernelGGL((m2l_bcast_kernel<P, NC, kBcastCos>), grid, blk, 0, s, a, L);
        BcastArgs b = a;  // the sin part's operators and partial sums
        b.rot = a.rot_sin;
        b.coax = a.coax_sin;
        if (a.n_split > 0) b.partial += a.n_partial * ((P + 1) * (P + 1) * 64);
        hipLaunchKernelGGL((m2l_bcast_kernel<P, NC, kBcastSin>), grid, blk, 0, s, b, L);
    } else {
        hipLaunchKernelGGL((m2l_bcast_kernel<P, NC, kBcastBoth>), grid, blk, 0, s, a, L);
    }
    if (a.n_split > 0) {
        const int64_t n = a.n_split * (P + 1) * (P + 1) * 64;
        hipLaunchKernelGGL((m2l_bcast_reduce_kernel<P, NC>), dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0,
                           s, a, L);
    }
}

template <int P>
void bcast_launch_nc(const BcastArgs& a, int nc, double* L, hipStream_t s)
{
    switch (nc) {
    case 1: bcast_launch<P, 1>(a, L, s); break;
    case 2: bcast_launch<P, 2>(a, L, s); break;
    case 3: bcast_launch<P, 3>(a, L, s); break;
    default: bcast_launch<P, 4>(a, L, s); break;
    }
}

}  // namespace

// Launches the kernel when p is one of Ps; false otherwise.
template <int... Ps>
bool bcast_dispatch(const BcastArgs& a, int p, int nc, double* L, hipStream_t s)
{
    bool done = false;
    ((p == Ps ? (bcast_launch_nc<Ps>(a, nc, L, s), done = true) : false), ...);
    return done;
}

}  // namespace sfmm
