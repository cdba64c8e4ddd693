// Half lengths N = N1·N2 of the wavefront x pass (sp_x2.hpp): for every N in
// 16..256 that splits into two radices of at most 16, the split with the
// smaller larger radix.  125, 162, 200, 216, 243 and 250 have none and stay
// with the block kernels.  X(N1, N2); two lists, one per compilation unit.
#pragma once

namespace dns {
// FP64 stops at N2 = 12: the registers of three components of 15 or 16 points
// per lane spill (450-540 B per lane).
template <typename T> constexpr bool sp_x2_shape(int n2) { return sizeof(T) == 4 || n2 <= 12; }
}  // namespace dns

#define SP_X2_SHAPES_LO \
    X(4, 4) \
    X(6, 3) \
    X(5, 4) \
    X(6, 4) \
    X(5, 5) \
    X(9, 3) \
    X(6, 5) \
    X(8, 4) \
    X(6, 6) \
    X(8, 5) \
    X(9, 5) \
    X(8, 6) \
    X(10, 5) \
    X(9, 6) \
    X(10, 6) \
    X(8, 8) \
    X(9, 8) \
    X(15, 5) \
    X(10, 8) \
    X(9, 9) \
    X(10, 9)

#define SP_X2_SHAPES_HI \
    X(12, 8) \
    X(10, 10) \
    X(12, 9) \
    X(12, 10) \
    X(16, 8) \
    X(15, 9) \
    X(12, 12) \
    X(15, 10) \
    X(16, 10) \
    X(15, 12) \
    X(16, 12) \
    X(15, 15) \
    X(16, 15) \
    X(16, 16)
