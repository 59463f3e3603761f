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

// fmod(|r|, b) with the sign of r, b > 0 (no difference would end the loop at
// 0) or NaN (r): exact as fmod is (each difference of two numbers within a
// factor of two is), in a few instructions a binary digit of |r| / b; NaN for an
// infinite r.  The library's loop costs a kernel some 20 registers.
template <typename T> LDL_HD T fmod_digits(T r, T b) {
    T a = fabs(r);
    if (!(a < T(INFINITY))) return T(NAN);
    while (a >= b) {
        T s = ldexp(b, ilogb(a) - ilogb(b));
        if (s > a) s *= T(0.5);
        a -= s;
    }
    return copysign(a, r);
}

// Period of an axis in T; NaN, which every mesh coordinate then is, for a box
// that rounds to zero (as with fmod; a test of b in fmod_digits costs its
// kernels up to 6 scalar registers, some a wavefront per SIMD).
template <typename T> inline T period_of(double box) {
    const T b = (T)box;
    return b > T(0) ? b : T(NAN);
}

// Mesh coordinate of the absolute position r: numpy remainder semantics, then
// division (jaxpops_bind.py:163-164).  fmod is the identity on [0, L), exactly
// r - L on [L, 2L) and the identity again on (-L, 0), where L is added.
template <typename T> LDL_HD T mesh_coordinate(T r, T box, T cell, T cellrcp) {
    if (!(r >= T(0) && r < box)) {
        if (r >= box && r < T(2) * box) r -= box;
        else if (!(r > -box && r < T(0))) r = fmod_digits(r, box);
        if (r < T(0)) r += box;
    }
    return div_by_cell(r, cell, cellrcp);
}

}  // namespace ldl
