#include "sp_x2_kernels.hpp"
#include "sp_x2_shapes.hpp"

namespace dns {

bool sp_x2_f64_lo(const X2Args<double> &a, int blocks, int waves, hipStream_t st)
{
#define X(A, B) \
    if (a.n == 2 * (A) * (B)) return sp_x2_go<double, A, B>(a, blocks, waves, st);
    SP_X2_SHAPES_LO
#undef X
    return false;
}

}  // namespace dns
