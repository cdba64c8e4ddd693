// Dispatch of the two-step pencil passes over their compilation units.
#include "p2.hpp"
#include "p2_shapes.hpp"

namespace dns {

bool p2_f32_0(int, const P2Args<float> &, dim3, hipStream_t);
bool p2_f32_1(int, const P2Args<float> &, dim3, hipStream_t);
bool p2_f32_2(int, const P2Args<float> &, dim3, hipStream_t);
bool p2_f32_3(int, const P2Args<float> &, dim3, hipStream_t);
bool p2_f64_0(int, const P2Args<double> &, dim3, hipStream_t);
bool p2_f64_1(int, const P2Args<double> &, dim3, hipStream_t);
bool p2_f64_2(int, const P2Args<double> &, dim3, hipStream_t);
bool p2_f64_3(int, const P2Args<double> &, dim3, hipStream_t);

bool p2_launch(P2Kind kind, const P2Args<float> &a, dim3 grid, hipStream_t st)
{
    return p2_f32_0(kind, a, grid, st) || p2_f32_1(kind, a, grid, st) || p2_f32_2(kind, a, grid, st) ||
           p2_f32_3(kind, a, grid, st);
}
bool p2_launch(P2Kind kind, const P2Args<double> &a, dim3 grid, hipStream_t st)
{
    return p2_f64_0(kind, a, grid, st) || p2_f64_1(kind, a, grid, st) || p2_f64_2(kind, a, grid, st) ||
           p2_f64_3(kind, a, grid, st);
}

template <typename T> bool p2_serves(P2Kind kind, int n)
{
#define X(A, B) \
    if (n == (A) * (B)) return kind != P2_STAGE || p2_stage_shape(A, B);
    P2_SHAPES_0
    P2_SHAPES_1
    P2_SHAPES_2
    P2_SHAPES_3
#undef X
    return false;
}
template bool p2_serves<float>(P2Kind, int);
template bool p2_serves<double>(P2Kind, int);

}  // namespace dns
