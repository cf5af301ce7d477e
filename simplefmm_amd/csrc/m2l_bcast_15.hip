// Broadcast M2L kernels, order 15.
#include "m2l_bcast_kernel.hpp"

namespace sfmm {

bool m2l_bcast_15(const BcastArgs& a, int p, int nc, double* L, hipStream_t s)
{
    return bcast_dispatch<15>(a, p, nc, L, s);
}

}  // namespace sfmm
