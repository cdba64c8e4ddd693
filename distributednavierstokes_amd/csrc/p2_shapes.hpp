// Line lengths n = N1·N2 of the two-step pencil passes (p2.hpp): every n in
// 24..512 of the factors 2, 3 and 5, split with the smaller larger radix.
// X(N1, N2); four lists, one per compilation unit.
#pragma once

#define P2_SHAPES_0 \
    X(6, 4) \
    X(8, 4) \
    X(8, 6) \
    X(8, 8) \
    X(9, 9) \
    X(12, 9) \
    X(15, 9) \
    X(18, 9) \
    X(18, 12) \
    X(25, 10) \
    X(20, 15) \
    X(25, 15) \
    X(24, 18) \
    X(25, 20)

#define P2_SHAPES_1 \
    X(5, 5) \
    X(6, 6) \
    X(10, 5) \
    X(9, 8) \
    X(10, 9) \
    X(12, 10) \
    X(12, 12) \
    X(15, 12) \
    X(15, 15) \
    X(16, 16) \
    X(20, 16) \
    X(24, 16) \
    X(25, 18) \
    X(32, 16)

#define P2_SHAPES_2 \
    X(9, 3) \
    X(8, 5) \
    X(9, 6) \
    X(15, 5) \
    X(12, 8) \
    X(25, 5) \
    X(15, 10) \
    X(16, 12) \
    X(16, 15) \
    X(18, 15) \
    X(18, 18) \
    X(20, 20) \
    X(24, 20)

#define P2_SHAPES_3 \
    X(6, 5) \
    X(9, 5) \
    X(10, 6) \
    X(10, 8) \
    X(10, 10) \
    X(16, 8) \
    X(16, 10) \
    X(20, 10) \
    X(27, 9) \
    X(18, 16) \
    X(20, 18) \
    X(27, 15) \
    X(27, 18)
