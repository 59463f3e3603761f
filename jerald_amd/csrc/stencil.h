// Real-space derivative stencils of the LDL layer on gfx950.
#pragma once

#include <algorithm>
#include <type_traits>

#include "ldl_common.h"

namespace ldl {

// ------------------------------------------- real-space derivative stencils
// The derivative symbol of k_axis_tables, D_d = (45 sin t - 9 sin 2t +
// sin 3t) / (30 h_d) with t = 2 pi n / N_d, is that of the 6th-order central
// difference
//   diff_d(a)[x] = 45 (a[x+1] - a[x-1]) - 9 (a[x+2] - a[x-2]) + (a[x+3] - a[x-3])
// along axis d (circular): a circular shift by s multiplies transform bin n
// by exp(+-2 pi i n s / N), so the transform of diff_d(a) / (60 h_d) is
// i D_d times the transform of a, and the inverse transform of -i D_d P is
// -diff_d(phi) / (60 h_d) with phi the inverse transform of P.  A layer on a
// power-of-two mesh therefore transforms one mesh each way: k_grad6 turns the potential phi
// into the forces F_d = -diff_d(phi) / (60 h_d), and k_div6 turns the
// painted gradient meshes g_d into sum_d diff_d(g_d) / (60 h_d), whose
// transform is the sum_d i D_d of theirs.
//
// Marching kernels: a workgroup of 4 TZ threads covers kStTY (y) x TZ (z) cells
// (each thread 4 cells along y at one z) and marches through xc x planes: the x
// difference comes from a 7-plane register queue per cell, the y and z
// differences from the current plane staged in LDS with 3-cell halos.  All
// indices are wrapped, so a tile larger than the mesh reads valid periodic
// values and only its stores are bounded.
constexpr int kStTY = 16;
// Widest tile: its 3-cell z halo costs two extra cache lines per row, so
// wider rows fetch less (FP32, 512^3: grad6 0.462 -> 0.437 ms, div6 0.482 ->
// 0.411 ms from 64 to 256); FP64 stops at 128 (at 1024 threads its divergence
// would spill)
template <typename T> constexpr int st_tz_max() { return sizeof(T) == 4 ? 256 : 128; }

struct StGeom {
    int n0, n1, n2, tiles_y, tiles_z, chunks, xc;
};

__device__ __forceinline__ int st_wrap(int v, int n) { return ((v % n) + n) % n; }

template <typename T>
__device__ __forceinline__ T st_diff(T m3, T m2, T m1, T p1, T p2, T p3) {
    return T(45) * (p1 - m1) - T(9) * (p2 - m2) + (p3 - m3);
}

template <int TZ> struct StTile {
    int x0, x1, y0, z0, tz, yg;
    int zw, yw[4];
    bool zok, yok[4];
    // halo cells this thread stages: y-halo rows hy[0..1] (row index of the
    // (kStTY + 6)-row plane, -1 none) at its own z; one z-halo cell (zrow, zcol)
    int hy[2], hyw[2], zrow, zcol, zyw, zzw;
    __device__ __forceinline__ StTile(const StGeom& g) {
        const int t = (int)xcd_tile(blockIdx.x, gridDim.x);
        const int tzt = t % g.tiles_z, tyt = (t / g.tiles_z) % g.tiles_y, xc = t / (g.tiles_z * g.tiles_y);
        x0 = xc * g.xc;
        x1 = x0 + g.xc < g.n0 ? x0 + g.xc : g.n0;
        y0 = tyt * kStTY;
        z0 = tzt * TZ;
        tz = threadIdx.x % TZ;
        yg = threadIdx.x / TZ;
        zw = st_wrap(z0 + tz, g.n2);
        zok = z0 + tz < g.n2;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int y = y0 + 4 * yg + c;
            yw[c] = st_wrap(y, g.n1);
            yok[c] = y < g.n1;
        }
        // y halo: rows 0..2 and kStTY+3..kStTY+5; thread rows yg and yg + 4
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int r = yg + 4 * h;
            hy[h] = r < 6 ? (r < 3 ? r : kStTY + r) : -1;
            hyw[h] = st_wrap(y0 + (hy[h] < 0 ? 0 : hy[h]) - 3, g.n1);
        }
        // z halo: kStTY rows x 6 columns (0..2, TZ+3..TZ+5), threads 0..95
        const int tt = threadIdx.x;
        zrow = tt < 6 * kStTY ? tt / 6 : -1;
        const int k = tt - (tt / 6) * 6;
        zcol = k < 3 ? k : TZ + k;
        zyw = st_wrap(y0 + (zrow < 0 ? 0 : zrow), g.n1);
        zzw = st_wrap(z0 + zcol - 3, g.n2);
    }
};

// Forces F (N0, N1, N2, 3), interleaved per cell, from the potential phi.
template <typename T, int TZ>
__global__ void __launch_bounds__(4 * TZ) k_grad6(const T* __restrict__ phi, T* __restrict__ F, StGeom g, T cx, T cy, T cz) {
    __shared__ T pl[kStTY + 6][TZ + 6];
    const StTile<TZ> tl(g);
    if (tl.x0 >= g.n0) return;  // uniform over the workgroup
    const int64_t ps = (int64_t)g.n1 * g.n2;
    auto at = [&](int x, int y, int z) { return phi[(int64_t)st_wrap(x, g.n0) * ps + (int64_t)y * g.n2 + z]; };
    T q[4][7];
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int k = 0; k < 7; k++) q[c][k] = at(tl.x0 - 3 + k, tl.yw[c], tl.zw);
    T hy0 = at(tl.x0, tl.hyw[0], tl.zw), hy1 = tl.hy[1] >= 0 ? at(tl.x0, tl.hyw[1], tl.zw) : T(0);
    T hz = tl.zrow >= 0 ? at(tl.x0, tl.zyw, tl.zzw) : T(0);
    for (int x = tl.x0; x < tl.x1; x++) {
        __syncthreads();  // the previous plane's reads are done
#pragma unroll
        for (int c = 0; c < 4; c++) pl[4 * tl.yg + c + 3][tl.tz + 3] = q[c][3];
        pl[tl.hy[0]][tl.tz + 3] = hy0;
        if (tl.hy[1] >= 0) pl[tl.hy[1]][tl.tz + 3] = hy1;
        if (tl.zrow >= 0) pl[tl.zrow + 3][tl.zcol] = hz;
        __syncthreads();
        // next plane's halo and the queue head, in flight during this plane
        T head[4];
        const bool more = x + 1 < tl.x1;
        if (more) {
#pragma unroll
            for (int c = 0; c < 4; c++) head[c] = at(x + 4, tl.yw[c], tl.zw);
            hy0 = at(x + 1, tl.hyw[0], tl.zw);
            if (tl.hy[1] >= 0) hy1 = at(x + 1, tl.hyw[1], tl.zw);
            if (tl.zrow >= 0) hz = at(x + 1, tl.zyw, tl.zzw);
        }
        if (tl.zok) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
                if (!tl.yok[c]) continue;
                const int ly = 4 * tl.yg + c + 3, lz = tl.tz + 3;
                const T dx = st_diff(q[c][0], q[c][1], q[c][2], q[c][4], q[c][5], q[c][6]);
                const T dy = st_diff(pl[ly - 3][lz], pl[ly - 2][lz], pl[ly - 1][lz], pl[ly + 1][lz], pl[ly + 2][lz], pl[ly + 3][lz]);
                const T dz = st_diff(pl[ly][lz - 3], pl[ly][lz - 2], pl[ly][lz - 1], pl[ly][lz + 1], pl[ly][lz + 2], pl[ly][lz + 3]);
                T* o = F + 3 * ((int64_t)x * ps + (int64_t)(tl.y0 + 4 * tl.yg + c) * g.n2 + (tl.z0 + tl.tz));
                o[0] = -cx * dx;
                o[1] = -cy * dy;
                o[2] = -cz * dz;
            }
        }
        if (more) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
#pragma unroll
                for (int k = 0; k < 6; k++) q[c][k] = q[c][k + 1];
                q[c][6] = head[c];
            }
        }
    }
}

// Divergence out = sum_d c_d diff_d(g_d) of the meshes g (3 consecutive
// (N0, N1, N2) meshes) into a real mesh.
template <typename T, int TZ>
__global__ void __launch_bounds__(4 * TZ) k_div6(const T* __restrict__ gm, T* __restrict__ out, StGeom g, T cx, T cy, T cz) {
    __shared__ T ly_[kStTY + 6][TZ];
    __shared__ T lz_[kStTY][TZ + 6];
    const StTile<TZ> tl(g);
    if (tl.x0 >= g.n0) return;  // uniform over the workgroup
    const int64_t ps = (int64_t)g.n1 * g.n2, cells = ps * g.n0;
    const T* gx = gm;
    const T* gy = gm + cells;
    const T* gz = gm + 2 * cells;
    auto at = [&](const T* a, int x, int y, int z) { return a[(int64_t)st_wrap(x, g.n0) * ps + (int64_t)y * g.n2 + z]; };
    T q[4][7], vy[4], vz[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
#pragma unroll
        for (int k = 0; k < 7; k++) q[c][k] = at(gx, tl.x0 - 3 + k, tl.yw[c], tl.zw);
        vy[c] = at(gy, tl.x0, tl.yw[c], tl.zw);
        vz[c] = at(gz, tl.x0, tl.yw[c], tl.zw);
    }
    T hy0 = at(gy, tl.x0, tl.hyw[0], tl.zw), hy1 = tl.hy[1] >= 0 ? at(gy, tl.x0, tl.hyw[1], tl.zw) : T(0);
    T hz = tl.zrow >= 0 ? at(gz, tl.x0, tl.zyw, tl.zzw) : T(0);
    for (int x = tl.x0; x < tl.x1; x++) {
        __syncthreads();  // the previous plane's reads are done
#pragma unroll
        for (int c = 0; c < 4; c++) {
            ly_[4 * tl.yg + c + 3][tl.tz] = vy[c];
            lz_[4 * tl.yg + c][tl.tz + 3] = vz[c];
        }
        ly_[tl.hy[0]][tl.tz] = hy0;
        if (tl.hy[1] >= 0) ly_[tl.hy[1]][tl.tz] = hy1;
        if (tl.zrow >= 0) lz_[tl.zrow][tl.zcol] = hz;
        __syncthreads();
        T head[4];
        const bool more = x + 1 < tl.x1;
        if (more) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
                head[c] = at(gx, x + 4, tl.yw[c], tl.zw);
                vy[c] = at(gy, x + 1, tl.yw[c], tl.zw);
                vz[c] = at(gz, x + 1, tl.yw[c], tl.zw);
            }
            hy0 = at(gy, x + 1, tl.hyw[0], tl.zw);
            if (tl.hy[1] >= 0) hy1 = at(gy, x + 1, tl.hyw[1], tl.zw);
            if (tl.zrow >= 0) hz = at(gz, x + 1, tl.zyw, tl.zzw);
        }
        if (tl.zok) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
                if (!tl.yok[c]) continue;
                const int r = 4 * tl.yg + c, z = tl.tz;
                const T dx = st_diff(q[c][0], q[c][1], q[c][2], q[c][4], q[c][5], q[c][6]);
                const T dy = st_diff(ly_[r][z], ly_[r + 1][z], ly_[r + 2][z], ly_[r + 4][z], ly_[r + 5][z], ly_[r + 6][z]);
                const T dz = st_diff(lz_[r][z], lz_[r][z + 1], lz_[r][z + 2], lz_[r][z + 4], lz_[r][z + 5], lz_[r][z + 6]);
                out[(int64_t)x * ps + (int64_t)(tl.y0 + r) * g.n2 + (tl.z0 + z)] = cx * dx + cy * dy + cz * dz;
            }
        }
        if (more) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
#pragma unroll
                for (int k = 0; k < 6; k++) q[c][k] = q[c][k + 1];
                q[c][6] = head[c];
            }
        }
    }
}

// Direct kernels: one cell per thread, its 18 neighbours read through the
// caches.
struct StCell {
    uint32_t x, y, z;
    __device__ __forceinline__ StCell(uint32_t i, const StGeom& g) {
        z = i % (uint32_t)g.n2;
        const uint32_t r = i / (uint32_t)g.n2;
        y = r % (uint32_t)g.n1;
        x = r / (uint32_t)g.n1;
    }
};
// circular neighbours v + k, k = -3..3 without 0, of v < n (n >= 3: one wrap)
__device__ __forceinline__ void st_ring(uint32_t v, uint32_t n, uint32_t (&w)[6]) {
#pragma unroll
    for (int k = 0; k < 6; k++) {
        int t = (int)v + (k < 3 ? k - 3 : k - 2);
        if (t < 0) t += (int)n;
        if (t >= (int)n) t -= (int)n;
        w[k] = (uint32_t)t;
    }
}
template <typename T>
__device__ __forceinline__ T st_ring_diff(const T* __restrict__ a, uint32_t base, const uint32_t (&w)[6], uint32_t stride) {
    return st_diff(a[base + w[0] * stride], a[base + w[1] * stride], a[base + w[2] * stride], a[base + w[3] * stride], a[base + w[4] * stride],
                   a[base + w[5] * stride]);
}

template <typename T>
__global__ void __launch_bounds__(256) k_grad6_direct(const T* __restrict__ phi, T* __restrict__ F, StGeom g, uint32_t cells, T cx, T cy, T cz) {
    const uint32_t i = (uint32_t)xcd_tile(blockIdx.x, gridDim.x) * 256u + threadIdx.x;
    if (i >= cells) return;
    const StCell c(i, g);
    const uint32_t sy = (uint32_t)g.n2, sx = (uint32_t)g.n1 * sy;
    uint32_t wx[6], wy[6], wz[6];
    st_ring(c.x, (uint32_t)g.n0, wx);
    st_ring(c.y, (uint32_t)g.n1, wy);
    st_ring(c.z, (uint32_t)g.n2, wz);
    const T dx = st_ring_diff(phi, i - c.x * sx, wx, sx), dy = st_ring_diff(phi, i - c.y * sy, wy, sy), dz = st_ring_diff(phi, i - c.z, wz, 1u);
    T* o = F + 3 * (int64_t)i;
    o[0] = -cx * dx;
    o[1] = -cy * dy;
    o[2] = -cz * dz;
}

template <typename T>
__global__ void __launch_bounds__(256) k_div6_direct(const T* __restrict__ gm, T* __restrict__ out, StGeom g, uint32_t cells, T cx, T cy, T cz) {
    const uint32_t i = (uint32_t)xcd_tile(blockIdx.x, gridDim.x) * 256u + threadIdx.x;
    if (i >= cells) return;
    const StCell c(i, g);
    const uint32_t sy = (uint32_t)g.n2, sx = (uint32_t)g.n1 * sy;
    uint32_t wx[6], wy[6], wz[6];
    st_ring(c.x, (uint32_t)g.n0, wx);
    st_ring(c.y, (uint32_t)g.n1, wy);
    st_ring(c.z, (uint32_t)g.n2, wz);
    const T dx = st_ring_diff(gm, i - c.x * sx, wx, sx), dy = st_ring_diff(gm + cells, i - c.y * sy, wy, sy),
            dz = st_ring_diff(gm + 2 * (int64_t)cells, i - c.z, wz, 1u);
    out[i] = cx * dx + cy * dy + cz * dz;
}

template <typename T>
inline StGeom st_geom(const Mesh& m, int tz, int xc) {
    StGeom g;
    g.n0 = (int)m.n0;
    g.n1 = (int)m.n1;
    g.n2 = (int)m.n2;
    g.xc = xc;
    g.tiles_y = (int)((m.n1 + kStTY - 1) / kStTY);
    g.tiles_z = (int)((m.n2 + tz - 1) / tz);
    g.chunks = (int)((m.n0 + xc - 1) / xc);
    return g;
}

// Direct kernels up to 2^20 cells: the mesh sits in the L2s, and marching
// leaves most CUs without a workgroup (64^3 FP32: one 64-plane march of 4
// workgroups 100 and 109 us, the shortest march 6.9 and 7.0, direct 3.7 and
// 3.5; 100^3: march 9.8 and 9.2, direct 9.2 and 8.2; 128^3: march 10.5 and
// 9.6, direct 15.8 and 14.9).
constexpr int64_t kStDirect = 1 << 20;

// Marching tile and chunk: 64 cells wide below 2^24 cells (more, smaller
// workgroups), else the width that pads n2 least, the widest on a tie (FP32
// 384^3 grad6: 200 us at 128, 248 at 256); then the longest chunk of 64, 32,
// 16, 8 or 4 planes that still gives 256 workgroups and 512 threads per CU
// (256^3 FP64: 128 x 32 planes 110 and 114 us, 64 planes 179 and 170).
template <typename T>
inline StGeom st_plan(const Mesh& m, int* tz) {
    *tz = 64;
    if (m.cells() >= (int64_t(1) << 24)) {
        int64_t best = (m.n2 + 63) / 64 * 64;
        for (int w = 128; w <= st_tz_max<T>(); w *= 2) {
            const int64_t pad = (m.n2 + w - 1) / w * w;
            if (pad <= best) {
                best = pad;
                *tz = w;
            }
        }
    }
    int xc = 64;
    for (; xc > 4; xc /= 2) {
        const StGeom g = st_geom<T>(m, *tz, xc);
        const int64_t blocks = (int64_t)g.chunks * g.tiles_y * g.tiles_z;
        if (blocks >= 256 && blocks * *tz >= 256 * 128) break;
    }
    return st_geom<T>(m, *tz, xc);
}

template <typename T, class Direct, class March>
inline void st_launch(const Mesh& m, Direct&& direct, March&& march) {
    if (m.cells() <= kStDirect && std::min(m.n0, std::min(m.n1, m.n2)) >= 3) {
        direct(st_geom<T>(m, 64, 64), (unsigned)((m.cells() + 255) / 256));
        return;
    }
    int tz;
    const StGeom g = st_plan<T>(m, &tz);
    const unsigned nb = (unsigned)((int64_t)g.chunks * g.tiles_y * g.tiles_z);
    if (tz == 64) march(g, nb, std::integral_constant<int, 64>{});
    else if (tz == 128) march(g, nb, std::integral_constant<int, 128>{});
    else if constexpr (sizeof(T) == 4) march(g, nb, std::integral_constant<int, 256>{});
}

// F = -(cx diff_x, cy diff_y, cz diff_z) phi, interleaved per cell
template <typename T>
inline void launch_grad6(const Mesh& m, const T* phi, T* F, T cx, T cy, T cz, hipStream_t st) {
    KTimer _t("grad6", st);
    st_launch<T>(
        m,
        [&](const StGeom& g, unsigned nb) {
            hipLaunchKernelGGL(k_grad6_direct<T>, dim3(nb), dim3(256), 0, st, phi, F, g, (uint32_t)m.cells(), cx, cy, cz);
        },
        [&](const StGeom& g, unsigned nb, auto TZ) {
            hipLaunchKernelGGL((k_grad6<T, decltype(TZ)::value>), dim3(nb), dim3(4 * decltype(TZ)::value), 0, st, phi, F, g, cx, cy, cz);
        });
}

// out = cx diff_x g_0 + cy diff_y g_1 + cz diff_z g_2 of three consecutive meshes
template <typename T>
inline void launch_div6(const Mesh& m, const T* gm, T* out, T cx, T cy, T cz, hipStream_t st) {
    KTimer _t("div6", st);
    st_launch<T>(
        m,
        [&](const StGeom& g, unsigned nb) {
            hipLaunchKernelGGL(k_div6_direct<T>, dim3(nb), dim3(256), 0, st, gm, out, g, (uint32_t)m.cells(), cx, cy, cz);
        },
        [&](const StGeom& g, unsigned nb, auto TZ) {
            hipLaunchKernelGGL((k_div6<T, decltype(TZ)::value>), dim3(nb), dim3(4 * decltype(TZ)::value), 0, st, gm, out, g, cx, cy, cz);
        });
}

}  // namespace ldl
