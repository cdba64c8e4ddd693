#include "p2_kernels.hpp"
#include "p2_shapes.hpp"

namespace dns {

bool p2_f64_2(int kind, const P2Args<double> &a, dim3 grid, hipStream_t st)
{
#define X(A, B) \
    if (a.n == (A) * (B)) return p2_go<double, A, B>(kind, a, grid, st);
    P2_SHAPES_2
#undef X
    return false;
}

}  // namespace dns
