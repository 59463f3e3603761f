// Arithmetic of the position decode: the remainder by the box size and the
// division by the cell size, in the working precision.
#pragma once

#include <cmath>

#ifndef LDL_HD
#define LDL_HD __device__ __forceinline__
#endif

namespace ldl {

// a / b, correctly rounded as the IEEE division, for positive normal b and y =
// RN(1 / b): two corrections of a y with exact residuals (Markstein, IBM J.
// Res. Dev. 34, 1990: one from a faithful quotient rounds correctly; the first
// makes it faithful).  Five operations instead of the division's dozen.  Tiny
// a, whose residuals could underflow, and y = 0 divide.
template <typename T> LDL_HD T div_by_cell(T a, T b, T y) {
    constexpr T tiny = sizeof(T) == 4 ? T(1e-25) : T(1e-250);
    if (!(a >= tiny) || y == T(0)) return a / b;
    T q = a * y;
    q = fma(fma(-b, q, a), y, q);
    return fma(fma(-b, q, a), y, q);
}

// fmod(|r|, b) with the sign of r, b >= 0: exact as fmod is (each difference of
// two numbers within a factor of two is), in a few instructions a binary digit
// of |r| / b; NaN for an infinite r and for b = 0 (a box too small for T), where
// no difference would end the loop.  The library's loop costs a kernel some 20
// registers.
template <typename T> LDL_HD T fmod_digits(T r, T b) {
    T a = fabs(r);
    if (!(a < T(INFINITY) && b > T(0))) return T(NAN);
    while (a >= b) {
        T s = ldexp(b, ilogb(a) - ilogb(b));
        if (s > a) s *= T(0.5);
        a -= s;
    }
    return copysign(a, r);
}

}  // namespace ldl
