// L2L kernels on matrix cores, orders 14..16.
#include "translate_mfma.hpp"

namespace sfmm {

bool translate_upper_top(const TransArgs& a, LevelSpan b, int p, int nc, double* io, hipStream_t s)
{
    return translate_dispatch<true, 14, 15, 16>(a, b, p, nc, io, s);
}

}  // namespace sfmm
