"""pow64.h's powers and logarithm, compiled for the CPU, against 113-bit ones:
within 0.56 + |a ln x| / 1024 ulp and 0.501 ulp (the roundings of the result
and of its last sums, and the logarithm's 2^-63 times the exponent).  Bases over
the density's range, within a factor of two of 1 and next to 1, exponents that
give every |a ln x| up to the cut; beyond it, and for bases that are not
positive and normal, the split form has to step aside."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "jerald_amd", "csrc")

DRIVER = r"""
#define LDL_HD inline
#include "pow64.h"
#include <quadmath.h>
#include <cmath>
#include <cstdio>
#include <limits>
#include <random>
using namespace ldl;
static double ulps(double v, __float128 t) {
    const double a = std::fabs((double)t);
    return std::fabs((double)((v - t) / (std::nextafter(a, INFINITY) - a)));
}
int main() {
    std::mt19937_64 g(1);
    std::uniform_real_distribution<double> u(0, 1);
    int bad = 0;
    auto check = [&](double x, double a) {
        const LogPair l = log_pair(x);
        const double y = std::fabs(a * l.h), e = ulps(pow_from_log(l, a), powq(x, a)), el = x == 1 ? std::fabs(l.h) : ulps(l.h, logq(x));
        if (!pow_pair_ok(x, a * l.h)) return;
        if (!(e <= 0.56 + y / 1024 && el <= 0.501) && bad++ < 5) std::printf("x %a a %a: pow %g ulp, log %g ulp\n", x, a, e, el);
    };
    for (double t : {0.01, 0.1, 1., 4., 16., 64., 256., 512., 700.})
        for (int i = 0; i < 20000; i++)
            for (int kind = 0; kind < 3; kind++) {
                const double x = kind == 0 ? std::exp(-18 + 30 * u(g)) : kind == 1 ? 0.6 + 0.9 * u(g) : 1 + (u(g) - 0.5) * std::pow(2., -45 * u(g));
                if (x != 1) check(x, t * (1 - 0.5 * u(g)) * (u(g) < 0.5 ? -1 : 1) / std::log(x));
            }
    check(0x1.68b5d909f9c8bp+0, -0x1.d4006a020a389p+10);  // 1.08 ulp
    for (double x : {1.0, 2.0, 0.5, 1e-8, 0x1p-1022, 0x1.fffffffffffffp1023, 0x1.6a09e667f3bcdp-1, 0x1.6a09e667f3bccp-1})
        for (double a : {0.0, 1.0, -1.0, 0.5, 2.0, 1e-300, 0.3}) check(x, a);
    using L = std::numeric_limits<double>;
    for (double x : {0.0, -0.0, -1.0, 0x1p-1023, L::infinity(), L::quiet_NaN()}) bad += pow_pair_ok(x, 0.5);
    for (double y : {700.1, -700.1, L::infinity(), L::quiet_NaN()}) bad += pow_pair_ok(2.0, y);
    return bad ? 1 : 0;
}
"""


def test_split_powers_against_113_bits(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O2", "-std=gnu++17", "-w", "-ffp-contract=off", f"-I{CSRC}", str(src), "-o", str(exe), "-lquadmath"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
