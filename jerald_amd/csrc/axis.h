// Per-axis wavenumber tables of the LDL kernels.
#pragma once

#include "ldl_common.h"

namespace ldl {

// Wavenumbers k = 2 pi fftfreq(N, cell) (pmesh.py:174-186; the z axis keeps
// N/2+1 entries, so its last one is -pi/cell) and the 6th-order
// finite-difference gradient symbol (45 sin kD - 9 sin 2kD + sin 3kD)/(30 D)
// (model.py:200-201), evaluated in FP64, of the three axes one after the other.
template <typename T> struct AxisTabs {
    T* k[3];
    T* D[3];
    int64_t n[3], count[3];
    double cell[3];
    __host__ __device__ int64_t total() const { return count[0] + count[1] + count[2]; }
    __device__ __forceinline__ void entry(int64_t i) const {
        int d = 0;
        while (d < 2 && i >= count[d]) i -= count[d++];
        const int64_t m = 2 * i < n[d] ? i : i - n[d];  // fftfreq order, odd n included: 0..(n-1)/2, -(n-1)/2..-1
        const double th = 2.0 * (double)m / (double)n[d];  // k cell / pi
        k[d][i] = (T)(2.0 * M_PI * (double)m / ((double)n[d] * cell[d]));
        D[d][i] = (T)((45.0 * sinpi(th) - 9.0 * sinpi(2.0 * th) + sinpi(3.0 * th)) / (30.0 * cell[d]));
    }
};
template <typename T> __global__ void __launch_bounds__(256) k_axis_tables(AxisTabs<T> a) {
    const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (i < a.total()) a.entry(i);
}

}  // namespace ldl
