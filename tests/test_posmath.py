"""The position decode's remainder and division against the C library's fmod
and the IEEE division, compiled for the CPU: ordinary and extreme ratios,
subnormal and infinite arguments, and boxes that round to zero."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "jerald_amd", "csrc")

DRIVER = r"""
#include <cmath>
using std::copysign; using std::fabs; using std::fma; using std::ilogb; using std::ldexp;
#define LDL_HD inline
#include "posmath.h"
#include <cstdio>
#include <limits>
#include <random>
template <typename T> bool same(T a, T b) { return std::isnan(a) ? std::isnan(b) : a == b && std::signbit(a) == std::signbit(b); }
template <typename T> int check(const char* name) {
    using L = std::numeric_limits<T>;
    std::mt19937_64 g(1);
    std::uniform_real_distribution<double> u(-1, 1);
    int bad = 0;
    auto rem = [&](T r, T b) {
        if (!same(ldl::fmod_digits(r, b), std::fmod(r, b)) && bad++ < 5) std::printf("%s fmod(%a, %a)\n", name, (double)r, (double)b);
    };
    const T edge[] = {T(0), -T(0), T(1), L::min(), L::denorm_min(), L::max(), L::infinity(), L::quiet_NaN(), T(51.3), T(-409.6)};
    for (T r : edge)
        for (T b : edge)
            if (b > T(0) && b < L::infinity()) rem(r, b);
    for (double box : {51.3, 1e-46, 4e-324, 1e-40, 409.6})  // some round to zero in T
        for (T r : edge) {
            const T L = ldl::period_of<T>(box), cell = L / 20;
            T u = std::fmod(r, (T)box);
            if (u < T(0)) u += (T)box;
            const T got = ldl::mesh_coordinate(r, L, cell, cell > T(1e-12) ? T(1) / cell : T(0));
            if (!same(got, u / ((T)box / 20)) && bad++ < 5) std::printf("%s coordinate %a in %g\n", name, (double)r, box);
        }
    for (int i = 0; i < 200000; i++) {
        const T b = std::ldexp((T)(1.5 + 0.5 * u(g)), (int)(20 * u(g)));
        rem((T)(u(g) * std::pow(2.0, 60 * u(g))) * b, b);
        const T a = (T)std::pow(2.0, 20 * u(g)), c = (T)std::pow(2.0, 10 * u(g));
        if (!same(ldl::div_by_cell(a, c, T(1) / c), a / c) && bad++ < 5) std::printf("%s %a / %a\n", name, (double)a, (double)c);
    }
    return bad;
}
int main() { return check<float>("float") + check<double>("double") ? 1 : 0; }
"""


def test_remainder_and_division_of_positions(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
