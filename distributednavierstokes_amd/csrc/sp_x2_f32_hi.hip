#include "sp_x2_kernels.hpp"
#include "sp_x2_shapes.hpp"

namespace dns {

bool sp_x2_f32_hi(const X2Args<float> &a, int blocks, int waves, hipStream_t st)
{
#define X(A, B) \
    if (a.n == 2 * (A) * (B)) return sp_x2_go<float, A, B>(a, blocks, waves, st);
    SP_X2_SHAPES_HI
#undef X
    return false;
}

}  // namespace dns
