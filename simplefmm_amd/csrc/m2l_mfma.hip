// Dispatch of the offset-grouped MFMA M2L (kernels in m2l_mfma.hpp).
#include "m2l_mfma.hpp"

namespace sfmm {

void launch_m2l_mfma(const M2LArgs& a, int p, int nc, const double* M, double* L, hipStream_t s)
{
    if (a.n_block == 0) return;
    // orders 13..16; the mixed path of lower orders runs m2l_dense.hpp
    (void)m2l_f32_top(a, p, nc, M, L, s);
}

// one translation unit per order range keeps the builds parallel
bool m2l_bcast_lo(const BcastArgs& a, int p, int nc, double* L, hipStream_t s);
bool m2l_bcast_hi(const BcastArgs& a, int p, int nc, double* L, hipStream_t s);
bool m2l_bcast_top(const BcastArgs& a, int p, int nc, double* L, hipStream_t s);
bool m2l_bcast_14(const BcastArgs& a, int p, int nc, double* L, hipStream_t s);
bool m2l_bcast_15(const BcastArgs& a, int p, int nc, double* L, hipStream_t s);
bool m2l_bcast_16(const BcastArgs& a, int p, int nc, double* L, hipStream_t s);

void launch_m2l_bcast(const BcastArgs& a, int p, int nc, double* L, hipStream_t s)
{
    if (a.n_item == 0) return;
    (void)(m2l_bcast_lo(a, p, nc, L, s) || m2l_bcast_hi(a, p, nc, L, s) || m2l_bcast_top(a, p, nc, L, s) ||
           m2l_bcast_14(a, p, nc, L, s) || m2l_bcast_15(a, p, nc, L, s) || m2l_bcast_16(a, p, nc, L, s));
}

}  // namespace sfmm
