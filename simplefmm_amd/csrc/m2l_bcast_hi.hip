// Broadcast M2L kernels, orders 9, 10, 11.
#include "m2l_bcast_kernel.hpp"

namespace sfmm {

bool m2l_bcast_hi(const BcastArgs& a, int p, int nc, double* L, hipStream_t s)
{
    return bcast_dispatch<9, 10, 11>(a, p, nc, L, s);
}

}  // namespace sfmm
