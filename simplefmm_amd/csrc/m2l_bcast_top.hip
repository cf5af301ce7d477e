// Broadcast M2L kernels, orders 12, 13.
#include "m2l_bcast_kernel.hpp"

namespace sfmm {

bool m2l_bcast_top(const BcastArgs& a, int p, int nc, double* L, hipStream_t s)
{
    return bcast_dispatch<12, 13>(a, p, nc, L, s);
}

}  // namespace sfmm
