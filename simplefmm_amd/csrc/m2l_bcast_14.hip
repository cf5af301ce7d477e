// Broadcast M2L kernels, order 14.
#include "m2l_bcast_kernel.hpp"

namespace sfmm {

bool m2l_bcast_14(const BcastArgs& a, int p, int nc, double* L, hipStream_t s)
{
    return bcast_dispatch<14>(a, p, nc, L, s);
}

}  // namespace sfmm
