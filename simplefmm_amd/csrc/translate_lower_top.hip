// M2M kernels on matrix cores, orders 14..16.
#include "translate_mfma.hpp"

namespace sfmm {

bool translate_lower_top(const TransArgs& a, LevelSpan b, int p, int nc, double* io, hipStream_t s)
{
    return translate_dispatch<false, 14, 15, 16>(a, b, p, nc, io, s);
}

}  // namespace sfmm
