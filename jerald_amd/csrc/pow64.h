// FP64 x^a for several a from one logarithm.
//
// The FP64 layer passes that raise the density to gamma are bound by vector
// instructions, not by memory, with library calls (each pow forms its own
// extended logarithm; the gamma adjoint took two of them and a log).  Here
// ln x = h + l is formed once to about 2^-63 of itself and each power is one
// exponential of a (h + l).  The logarithm's error enters times |a ln x|: a power
// is within 0.56 + |a ln x| / 1024 ulp where |a ln x| <= 700 (largest measured:
// 0.57 ulp to |a ln x| = 128, 0.66 at 256, 1.08 at 700; the library's pow over
// the same arguments: 1.34 from 4 on, 1.18 at 1).  h alone is the rounded
// logarithm (0.501 ulp; the library's 0.65).  256^3: gamma adjoint 287 -> 144
// us, density spectrum 132 -> 115.  Arguments beyond that (zero, negative,
// subnormal, infinite and NaN bases, powers near overflow or underflow) take the
// library's pow.
//
//   x = 2^e m, m in [sqrt(1/2), sqrt(2)), s = (m - 1) / (m + 1):
//   ln m = 2 artanh s = 2 s + s^3 (2/3 + 2/5 s^2 + ...), |s| <= 0.172, the
//   quotient with its remainder (s + sl), the series to s^23 (next term below
//   2^-65 of the sum)
//   e^r: r = y - n ln 2, |r| <= 0.347, Taylor to r^13 (next term 2^-57.8 of 1)
// with ln 2 split so that the multiples of its first part are exact.
#pragma once

#ifndef LDL_HD
#define LDL_HD __device__ __forceinline__
#endif

// The error terms below are exact only if no product is fused into a sum that
// does not say so.
#define LDL_NO_CONTRACT _Pragma("clang fp contract(off)")

namespace ldl {

struct LogPair {
    double h, l;  // ln x = h + l
};

// A reciprocal to a few ulp: the quotient below carries its remainder.
LDL_HD double rcp_near(double d) {
#ifdef __HIP_DEVICE_COMPILE__
    double r = __builtin_amdgcn_rcp(d);
    r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
    return __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
#else
    return 1.0 / d;
#endif
}

static constexpr double kLn2Hi = 0x1.62e42fefa38p-1;        // 42 bits: n kLn2Hi is exact for |n| < 2^11
static constexpr double kLn2Lo = 0x1.ef35793c7673p-45;      // ln 2 - kLn2Hi

// ln x for positive normal x.
LDL_HD LogPair log_pair(double x) {
    LDL_NO_CONTRACT
#ifdef __HIP_DEVICE_COMPILE__
    int e = __builtin_amdgcn_frexp_exp(x);
    double m = __builtin_amdgcn_frexp_mant(x);  // [1/2, 1)
#else
    int e;
    double m = __builtin_frexp(x, &e);
#endif
    if (m < 0x1.6a09e667f3bcdp-1) {
        m *= 2.0;
        e -= 1;
    }
    const double z = m - 1.0;  // exact
    const double d = m + 1.0;
    const double dl = m - (d - 1.0);  // d + dl = m + 1
    const double r = rcp_near(d);
    const double s = z * r;
    const double sl = __builtin_fma(-s, dl, __builtin_fma(-s, d, z)) * r;
    const double u = s * s;
    double p = 2.0 / 23.0;
    p = __builtin_fma(p, u, 2.0 / 21.0);
    p = __builtin_fma(p, u, 2.0 / 19.0);
    p = __builtin_fma(p, u, 2.0 / 17.0);
    p = __builtin_fma(p, u, 2.0 / 15.0);
    p = __builtin_fma(p, u, 2.0 / 13.0);
    p = __builtin_fma(p, u, 2.0 / 11.0);
    p = __builtin_fma(p, u, 2.0 / 9.0);
    p = __builtin_fma(p, u, 2.0 / 7.0);
    p = __builtin_fma(p, u, 2.0 / 5.0);
    // v + vl = s^3, c + cl = the series' bracket, b + bl = their product
    const double ul = __builtin_fma(s, s, -u);
    const double v = s * u;
    const double vl = __builtin_fma(u, 3.0 * sl, __builtin_fma(s, ul, __builtin_fma(s, u, -v)));
    constexpr double k3 = 2.0 / 3.0, k3l = 0x1.5555555555555p-55;  // 2/3 = k3 + k3l
    const double up = u * p;
    const double c = k3 + up;
    const double cl = up - (c - k3) + k3l;
    const double b = v * c;
    const double bl = __builtin_fma(v, cl, __builtin_fma(vl, c, __builtin_fma(v, c, -b)));
    // e kLn2Hi + 2 s + b, exactly as h1 and what t and t1 hold: each sum's
    // first term is the larger one (or e = 0)
    const double en = (double)e;
    const double a = en * kLn2Hi, s2 = 2.0 * s;
    const double h0 = a + s2;
    const double t = e == 0 ? 0.0 : s2 - (h0 - a);
    const double h1 = h0 + b;
    const double t1 = b - (h1 - h0);
    const double l1 = t1 + (t + (bl + __builtin_fma(en, kLn2Lo, 2.0 * sl)));
    const double h = h1 + l1;
    return LogPair{h, l1 - (h - h1)};
}

// e^(h + l) for |h| < 708, |l| <= ulp(h).
LDL_HD double exp_pair(double h, double l) {
    LDL_NO_CONTRACT
    const double n = __builtin_rint(h * 0x1.71547652b82fep0);
    const double r = __builtin_fma(-n, kLn2Hi, h);  // exact
    const double rl0 = __builtin_fma(-n, kLn2Lo, l);
    const double rh = r + rl0;
    const double rl = rl0 - (rh - r);
    double q = 1.0 / 6227020800.0;
    q = __builtin_fma(q, rh, 1.0 / 479001600.0);
    q = __builtin_fma(q, rh, 1.0 / 39916800.0);
    q = __builtin_fma(q, rh, 1.0 / 3628800.0);
    q = __builtin_fma(q, rh, 1.0 / 362880.0);
    q = __builtin_fma(q, rh, 1.0 / 40320.0);
    q = __builtin_fma(q, rh, 1.0 / 5040.0);
    q = __builtin_fma(q, rh, 1.0 / 720.0);
    q = __builtin_fma(q, rh, 1.0 / 120.0);
    q = __builtin_fma(q, rh, 1.0 / 24.0);
    q = __builtin_fma(q, rh, 1.0 / 6.0);
    // 1 + rh = s + c and s + rh^2/2 = s2 + c2 (+ hl); the rest is below 2^-7
    const double s = 1.0 + rh;
    const double c = rh - (s - 1.0);
    const double hh = 0.5 * rh * rh;
    const double hl = __builtin_fma(0.5 * rh, rh, -hh);
    const double s2 = s + hh;
    const double c2 = hh - (s2 - s);
    const double w = __builtin_fma(q, rh * (2.0 * hh), __builtin_fma(rl, rh, c + rl + hl) + c2);
    return __builtin_ldexp(s2 + w, (int)n);
}

// Whether x^a may be formed as exp_pair(a ln x): x normal, |a h| <= 700.
LDL_HD bool pow_pair_ok(double x, double ah) { return x >= 0x1p-1022 && x <= 0x1.fffffffffffffp1023 && __builtin_fabs(ah) <= 700.0; }

// x^a from ln x = g.
LDL_HD double pow_from_log(LogPair g, double a) {
    LDL_NO_CONTRACT
    const double h = a * g.h;
    return exp_pair(h, __builtin_fma(a, g.l, __builtin_fma(a, g.h, -h)));
}

}  // namespace ldl
