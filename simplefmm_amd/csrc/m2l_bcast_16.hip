// Broadcast M2L kernels, order 16.
#include "m2l_bcast_kernel.hpp"

namespace sfmm {

bool m2l_bcast_16(const BcastArgs& a, int p, int nc, double* L, hipStream_t s)
{
    return bcast_dispatch<16>(a, p, nc, L, s);
}

}  // namespace sfmm
