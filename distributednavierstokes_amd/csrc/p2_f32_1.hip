#include "p2_kernels.hpp"
#include "p2_shapes.hpp"

namespace dns {

bool p2_f32_1(int kind, const P2Args<float> &a, dim3 grid, hipStream_t st)
{
#define X(A, B) \
    if (a.n == (A) * (B)) return p2_go<float, A, B>(kind, a, grid, st);
    P2_SHAPES_1
#undef X
    return false;
}

}  // namespace dns
