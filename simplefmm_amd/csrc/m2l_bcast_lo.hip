// Broadcast M2L kernels, orders 1, 2, 3, 4, 5, 6, 7, 8.
#include "m2l_bcast_kernel.hpp"

namespace sfmm {

bool m2l_bcast_lo(const BcastArgs& a, int p, int nc, double* L, hipStream_t s)
{
    return bcast_dispatch<1, 2, 3, 4, 5, 6, 7, 8>(a, p, nc, L, s);
}

}  // namespace sfmm
