// Batched FFTs of any length whose prime factors are 2, 3 and 5, for mesh
// axes that are not powers of two.  Same conventions and pass structure as
// fft_core.h (Stockham autosort in LDS, unnormalised, forward exp(-2 pi i/N)).
// The stage list (radices 8, 4, 2, 5, 3 in that order) is a runtime plan; two
// consecutive stages whose radices multiply to at most 16 run as one group in
// registers, so a transform of 384 = 8 8 (2 3) makes three LDS round trips in
// place.  What bounds a pass is the memory it moves, as for powers of two.
// Host helpers pick the power-of-two kernels when they apply.
#pragma once

#include <algorithm>

#include "fft_core.h"

namespace ldl {

// A group of one stage (rb = 1) or two (radices ra, then rb): nbg = n / (ra rb)
// butterflies per pencil, ns = product of the radices before it, mag =
// ceil(2^20 / ns) (j / ns = j mag >> 20 for j < 1024, ns <= 1024), ta and tb
// the twiddle steps n / (ns ra) and n / (ns ra rb).
struct AnyGroup {
    int ra, rb, nbg, ns, ta, tb;
    unsigned mag;
};
// tpp: threads per pencil, enough for every group at any_bpt() butterflies a thread.
struct AnyPlan {
    int n, ngrp, tpp;
    AnyGroup g[8];
};

// Butterflies of a radix-r group per thread: up to 16 values.
__host__ __device__ constexpr int any_bpt(int r) { return r > 8 ? 1 : 16 / r; }

// Radix list for n (8s first, then 4, 2, 5, 3), grouped for the fewest groups
// and then the fewest threads per pencil; false if n has another prime factor.
inline bool any_plan(int64_t n, AnyPlan* pl) {
    if (n < 2 || n > 1024) return false;
    int radix[16], nst = 0;
    int64_t r = n;
    for (int f : {8, 4, 2, 5, 3})
        while (r % f == 0) {
            radix[nst++] = f;
            r /= f;
        }
    if (r != 1) return false;
    // the consecutive pairs any_fft has code for (8 2 would fit too, but the
    // compiler contracts its products differently: other bits than apart)
    auto pair_ok = [](int a, int b) { return (b == 3 && a <= 5) || (a == 2 && b == 5); };
    auto tpp_of = [&](int R) { return (int)((n / R + any_bpt(R) - 1) / any_bpt(R)); };
    // best[i]: (groups, threads) of the stages from i on; two: whether i and i + 1 pair up
    int bg[17], bt[17];
    bool two[17];
    bg[nst] = 0;
    bt[nst] = 1;
    for (int i = nst - 1; i >= 0; i--) {
        bg[i] = bg[i + 1] + 1;
        bt[i] = std::max(bt[i + 1], tpp_of(radix[i]));
        two[i] = false;
        if (i + 1 < nst && pair_ok(radix[i], radix[i + 1])) {
            const int g2 = bg[i + 2] + 1, t2 = std::max(bt[i + 2], tpp_of(radix[i] * radix[i + 1]));
            if (g2 < bg[i] || (g2 == bg[i] && t2 < bt[i])) {
                bg[i] = g2;
                bt[i] = t2;
                two[i] = true;
            }
        }
    }
    pl->n = (int)n;
    pl->tpp = bt[0];
    pl->ngrp = 0;
    int ns = 1;
    for (int i = 0; i < nst;) {
        AnyGroup& g = pl->g[pl->ngrp++];
        g.ra = radix[i];
        g.rb = two[i] ? radix[i + 1] : 1;
        g.ns = ns;
        g.nbg = (int)n / (g.ra * g.rb);
        g.ta = (int)n / (ns * g.ra);
        g.tb = (int)n / (ns * g.ra * g.rb);
        g.mag = ((1u << 20) + ns - 1) / ns;
        ns *= g.ra * g.rb;
        i += two[i] ? 2 : 1;
    }
    return true;
}

// 3- and 5-point DFTs with w = exp(DIR 2 pi i / R).
template <int DIR, typename C> __device__ __forceinline__ void dft3(C* v) {
    using S = decltype(v[0].x);
    const S s3 = S(0.86602540378443864676372317075294);  // sin(2 pi / 3)
    const C a = cadd(v[1], v[2]), b = csub(v[1], v[2]);
    const C t = C{v[0].x - S(0.5) * a.x, v[0].y - S(0.5) * a.y};
    const C u = rot90<DIR>(C{s3 * b.x, s3 * b.y});
    v[0] = cadd(v[0], a);
    v[1] = cadd(t, u);
    v[2] = csub(t, u);
}

template <int DIR, typename C> __device__ __forceinline__ void dft5(C* v) {
    using S = decltype(v[0].x);
    const S c1 = S(0.30901699437494742410229341718282);   // cos(2 pi / 5)
    const S c2 = S(-0.80901699437494742410229341718282);  // cos(4 pi / 5)
    const S s1 = S(0.95105651629515357211643933337938);   // sin(2 pi / 5)
    const S s2 = S(0.58778525229247312916870595463907);   // sin(4 pi / 5)
    const C a1 = cadd(v[1], v[4]), a2 = cadd(v[2], v[3]);
    const C b1 = csub(v[1], v[4]), b2 = csub(v[2], v[3]);
    const C t1 = C{v[0].x + c1 * a1.x + c2 * a2.x, v[0].y + c1 * a1.y + c2 * a2.y};
    const C t2 = C{v[0].x + c2 * a1.x + c1 * a2.x, v[0].y + c2 * a1.y + c1 * a2.y};
    const C u1 = rot90<DIR>(C{s1 * b1.x + s2 * b2.x, s1 * b1.y + s2 * b2.y});
    const C u2 = rot90<DIR>(C{s2 * b1.x - s1 * b2.x, s2 * b1.y - s1 * b2.y});
    v[0] = cadd(v[0], cadd(a1, a2));
    v[1] = cadd(t1, u1);
    v[4] = csub(t1, u1);
    v[2] = cadd(t2, u2);
    v[3] = csub(t2, u2);
}

template <int R, int DIR, typename C> __device__ __forceinline__ void dft_any(C* v) {
    if constexpr (R == 3) dft3<DIR>(v);
    else if constexpr (R == 5) dft5<DIR>(v);
    else dft<R, DIR>(v);
}

// One group on the P pencils of lds (element n of pencil p at lds[n LS + p]).
// Butterfly jj reads elements jj + e nbg, e < RA RB, and writes (jj - k) RA RB
// + k + e ns with k = jj mod ns: the inputs and outputs of the RB stage-RA
// butterflies and the RA stage-RB butterflies between them, each with the
// twiddles its own stage has.
template <typename T, int DIR, int P, int RA, int RB>
__device__ __forceinline__ void any_group(c2<T>* lds, const c2<T>* tw, int tws, const AnyGroup& g, int tpp) {
    using C = c2<T>;
    constexpr int R = RA * RB, B = any_bpt(R), LS = P + 1;
    const int p = threadIdx.x % P;
    const int q = (int)threadIdx.x / P < tpp ? (int)threadIdx.x / P : 4096;  // threads past the last butterfly only wait
    C v[B][R];
#pragma unroll
    for (int b = 0; b < B; b++) {
        const int jj = q + b * tpp;
        if (jj < g.nbg) {
#pragma unroll
            for (int e = 0; e < R; e++) v[b][e] = lds[(jj + e * g.nbg) * LS + p];
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < B; b++) {
        const int jj = q + b * tpp;
        if (jj < g.nbg) {
            const int k = jj - (int)(((unsigned)jj * g.mag) >> 20) * g.ns;
#pragma unroll
            for (int rb = 0; rb < RB; rb++) {
                C t[RA];
#pragma unroll
                for (int r = 0; r < RA; r++) t[r] = v[b][rb + r * RB];
                if (g.ns > 1) {
#pragma unroll
                    for (int r = 1; r < RA; r++) {
                        C w = tw[r * k * g.ta * tws];
                        if (DIR > 0) w.y = -w.y;
                        t[r] = cmul(t[r], w);
                    }
                }
                dft_any<RA, DIR>(t);
#pragma unroll
                for (int r = 0; r < RA; r++) v[b][rb + r * RB] = t[r];
            }
            const int base = (jj - k) * R + k;
#pragma unroll
            for (int ra = 0; ra < RA; ra++) {
                C t[RB];
#pragma unroll
                for (int r = 0; r < RB; r++) t[r] = v[b][r + ra * RB];
                if constexpr (RB > 1) {
#pragma unroll
                    for (int r = 1; r < RB; r++) {
                        C w = tw[r * (k + ra * g.ns) * g.tb * tws];
                        if (DIR > 0) w.y = -w.y;
                        t[r] = cmul(t[r], w);
                    }
                    dft_any<RB, DIR>(t);
                }
#pragma unroll
                for (int r = 0; r < RB; r++) lds[(base + (ra + r * RA) * g.ns) * LS + p] = t[r];
            }
        }
    }
    __syncthreads();
}

// Transform the P pencils of lds in place.  tw[m tws] = exp(-2 pi i m / n).
// All threads of the workgroup take part.
template <typename T, int DIR, int P>
__device__ __forceinline__ void any_fft(c2<T>* lds, const c2<T>* tw, int tws, const AnyPlan& pl) {
    for (int i = 0; i < pl.ngrp; i++) {
        const AnyGroup g = pl.g[i];
        switch (g.ra * 8 + g.rb) {
            case 8 * 8 + 1: any_group<T, DIR, P, 8, 1>(lds, tw, tws, g, pl.tpp); break;
            case 4 * 8 + 1: any_group<T, DIR, P, 4, 1>(lds, tw, tws, g, pl.tpp); break;
            case 4 * 8 + 3: any_group<T, DIR, P, 4, 3>(lds, tw, tws, g, pl.tpp); break;
            case 2 * 8 + 1: any_group<T, DIR, P, 2, 1>(lds, tw, tws, g, pl.tpp); break;
            case 2 * 8 + 5: any_group<T, DIR, P, 2, 5>(lds, tw, tws, g, pl.tpp); break;
            case 2 * 8 + 3: any_group<T, DIR, P, 2, 3>(lds, tw, tws, g, pl.tpp); break;
            case 5 * 8 + 1: any_group<T, DIR, P, 5, 1>(lds, tw, tws, g, pl.tpp); break;
            case 5 * 8 + 3: any_group<T, DIR, P, 5, 3>(lds, tw, tws, g, pl.tpp); break;
            case 3 * 8 + 1: any_group<T, DIR, P, 3, 1>(lds, tw, tws, g, pl.tpp); break;
            default: any_group<T, DIR, P, 3, 3>(lds, tw, tws, g, pl.tpp); break;
        }
    }
}

// i / d for i < 2^14, d <= 2^10, from m = ceil(2^32 / d) (1 < d).
__device__ __forceinline__ int div_by(int i, unsigned m) { return (int)__umulhi((unsigned)i, m); }
__host__ __device__ inline unsigned div_magic(unsigned d) { return (unsigned)(((1ull << 32) + d - 1) / d); }

// Launch shape of an any-length pass: P pencils, th threads, lds bytes.
struct AnyShape {
    int P, th;
    size_t lds;
};
// ``len`` LDS elements per pencil, a twiddle table of ``tlen``.  16 (FP64: 8)
// pencils are whole 128-byte lines of a column strip; half of that where two
// workgroups of at most 512 threads then fit a CU and did not before.  A pass
// of ``pencils`` pencils that leaves CUs idle gets a thread per butterfly
// (shorter chains), else the fewest threads (pl->tpp).
template <typename T>
inline AnyShape any_shape(AnyPlan* pl, int len, int tlen, int64_t pencils) {
    constexpr int PM = sizeof(T) == 4 ? 16 : 8;
    constexpr size_t half = 80 * 1024;
    auto shape = [&](int P) {
        return AnyShape{P, (P * pl->tpp + 63) / 64 * 64, ((size_t)len * (P + 1) + tlen) * sizeof(c2<T>)};
    };
    const AnyShape a = shape(PM), b = shape(PM / 2);
    AnyShape s = a;
    if (!(a.lds <= half && a.th <= 512) && (b.lds <= half || a.th > 1024 || a.lds > 2 * half)) s = b;
    if (pencils <= 512 * s.P) {
        int t = pl->tpp;
        for (int i = 0; i < pl->ngrp; i++) t = std::max(t, pl->g[i].nbg);
        pl->tpp = std::max(pl->tpp, std::min(t, 512 / s.P));
        s = shape(s.P);
    }
    return s;
}
// Dynamic LDS above 64 KB must be enabled per kernel.
template <typename K>
inline void allow_lds(K* kernel, size_t bytes) {
    if (bytes > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

template <typename T, int DIR, int P, class Op>
__global__ void __launch_bounds__(1024) k_colpass_any(ColGeom g, const c2<T>* __restrict__ tw, AnyPlan pl, Op op) {
    using C = c2<T>;
    extern __shared__ __align__(16) unsigned char any_smem[];
    constexpr int LS = P + 1, NV = 16;
    const int n = pl.n, nq = (int)blockDim.x / P;  // nq >= tpp >= n / 16
    C* a = reinterpret_cast<C*>(any_smem);
    C* twl = a + n * LS;
    const int64_t tile = xcd_tile_rev(blockIdx.x, gridDim.x);
    const int64_t plane = tile / g.tiles_per_plane;
    const int64_t col0 = (tile - plane * g.tiles_per_plane) * P;
    const int64_t base = plane * g.plane_stride + col0;
    const int pv = (int)((g.ncols - col0) < P ? (g.ncols - col0) : P);
    const int p = threadIdx.x % P, q = threadIdx.x / P, pc = p < pv ? p : pv - 1;
    for (int i = threadIdx.x; i < n; i += blockDim.x) twl[i] = tw[i];
    C v[NV];  // all of a thread's loads before the first LDS write
#pragma unroll
    for (int s = 0; s < NV; s++) {
        const int nn = q + s * nq;
        if (nn < n) v[s] = op.load(base + nn * g.es + pc, nn, plane, col0 + pc);
    }
#pragma unroll
    for (int s = 0; s < NV; s++) {
        const int nn = q + s * nq;
        if (nn < n) a[nn * LS + p] = p < pv ? v[s] : C{T(0), T(0)};
    }
    __syncthreads();
    any_fft<T, DIR, P>(a, twl, 1, pl);
    if (p < pv)
        for (int nn = q; nn < n; nn += nq) op.store(base + nn * g.es + p, nn, plane, col0 + p, a[nn * LS + p]);
}

// Real rows of N2 = 2H -> half spectrum (pl is the plan of H; tw2 the N2 table).
template <typename T, int P, class Pro, class Epi>
__global__ void __launch_bounds__(1024) k_zpass_r2c_any(int64_t nrows, const c2<T>* __restrict__ tw2, AnyPlan pl, Pro pro, Epi epi) {
    using C = c2<T>;
    extern __shared__ __align__(16) unsigned char any_smem[];
    constexpr int LS = P + 1;
    const int H = pl.n, N2 = 2 * H;
    C* a = reinterpret_cast<C*>(any_smem);
    C* twl = a + H * LS;
    const int64_t row0 = xcd_tile(blockIdx.x, gridDim.x) * (int64_t)P;
    for (int i = threadIdx.x; i < N2; i += blockDim.x) twl[i] = tw2[i];
    const unsigned mh = div_magic(H), mh1 = div_magic(H + 1);
    constexpr int NV = 16;  // blockDim >= H P / 16
    C v[NV];
#pragma unroll
    for (int s = 0; s < NV; s++) {
        const int i = threadIdx.x + s * blockDim.x;
        if (i < H * P) {
            const int p = div_by(i, mh), m = i - p * H;
            v[s] = pro.load2(row0 + p < nrows ? row0 + p : nrows - 1, m);
        }
    }
#pragma unroll
    for (int s = 0; s < NV; s++) {
        const int i = threadIdx.x + s * blockDim.x;
        if (i < H * P) {
            const int p = div_by(i, mh), m = i - p * H;
            a[m * LS + p] = row0 + p < nrows ? v[s] : C{T(0), T(0)};
        }
    }
    __syncthreads();
    any_fft<T, -1, P>(a, twl, 2, pl);
    for (int i = threadIdx.x; i < (H + 1) * P; i += blockDim.x) {
        const int p = div_by(i, mh1), k = i - p * (H + 1);
        if (row0 + p >= nrows) continue;
        const C zk = a[(k == H ? 0 : k) * LS + p];
        const C zc = cconj(a[(k == 0 ? 0 : H - k) * LS + p]);
        // E = (Z[k] + conj Z[H-k]) / 2, O = (Z[k] - conj Z[H-k]) / (2i), X = E + W^k O
        const C e = C{T(0.5) * (zk.x + zc.x), T(0.5) * (zk.y + zc.y)};
        const C d = csub(zk, zc);
        const C o = C{T(0.5) * d.y, T(-0.5) * d.x};
        epi.store(row0 + p, k, cadd(e, cmul(o, twl[k])));
    }
}

// block_sum for a runtime workgroup size (a multiple of 64, at most 1024);
// red holds NR * 16 values.
template <int NR>
__device__ __forceinline__ void block_sum_any(double (&v)[NR], double* red) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const double x = wave_sum(v[r]);
        if (lane == 0) red[r * 16 + w] = x;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int r = 0; r < NR; r++) {
            double x = 0.0;
            for (int i = 0; i < nw; i++) x += red[r * 16 + i];
            v[r] = x;
        }
    }
}
template <class Epi, int P> constexpr int any_rows() { return epi_triple<Epi>::value ? P / 3 * 3 : P; }

// Half spectrum rows -> real rows of N2 = 2H, with the Epi::NR reductions of
// k_zpass_c2r (workgroup totals to Epi::reduce_out(blockIdx.x, ...)).  Bins k
// and H - k are loaded together and both half-length inputs formed from them.
template <typename T, int P, class Pro, class Epi>
__global__ void __launch_bounds__(1024) k_zpass_c2r_any(int64_t nrows, const c2<T>* __restrict__ tw2, AnyPlan pl, Pro pro, Epi epi) {
    using C = c2<T>;
    extern __shared__ __align__(16) unsigned char any_smem[];
    constexpr int LS = P + 1, RPB = any_rows<Epi, P>();
    const int H = pl.n, N2 = 2 * H;
    C* a = reinterpret_cast<C*>(any_smem);
    C* twl = a + H * LS;
    const int64_t row0 = xcd_tile(blockIdx.x, gridDim.x) * (int64_t)RPB;
    for (int i = threadIdx.x; i < N2; i += blockDim.x) twl[i] = tw2[i];
    __syncthreads();
    const int HP = H / 2 + 1;
    const unsigned mp = div_magic(HP), mh = div_magic(H);
    constexpr int U = 4;  // pairs in flight per thread
    for (int i0 = threadIdx.x; i0 < HP * RPB; i0 += U * blockDim.x) {
        C xk[U], xc[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = i0 + u * blockDim.x;
            if (i < HP * RPB) {
                const int p = div_by(i, mp), k = i - p * HP;
                const int64_t row = row0 + p < nrows ? row0 + p : nrows - 1;
                xk[u] = pro.load(row, k);
                xc[u] = pro.load(row, H - k);
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = i0 + u * blockDim.x;
            if (i < HP * RPB) {
                const int p = div_by(i, mp), k = i - p * HP;
                if (k == 0) xk[u].y = xc[u].y = T(0);  // FFTW ignores these imaginary parts
                // Z'[k] = (X[k] + conj X[H-k]) + i (X[k] - conj X[H-k]) e^{+2 pi i k / N2}
                C t = twl[k];
                t.y = -t.y;
                const C e = cadd(xk[u], cconj(xc[u])), o = cmul(csub(xk[u], cconj(xc[u])), t);
                a[k * LS + p] = cadd(e, C{-o.y, o.x});
                if (k != 0 && 2 * k != H) {
                    C t2 = twl[H - k];
                    t2.y = -t2.y;
                    const C e2 = cadd(xc[u], cconj(xk[u])), o2 = cmul(csub(xc[u], cconj(xk[u])), t2);
                    a[(H - k) * LS + p] = cadd(e2, C{-o2.y, o2.x});
                }
            }
        }
    }
    __syncthreads();
    any_fft<T, +1, P>(a, twl, 2, pl);
    constexpr int NR = Epi::NR;
    double acc[NR > 0 ? NR : 1] = {};
    constexpr int RW = epi_triple<Epi>::value ? 3 : 1;  // rows a thread stores together
    for (int i = threadIdx.x; i < H * (RPB / RW); i += blockDim.x) {
        const int p = div_by(i, mh) * RW, m = i - p / RW * H;
        if (row0 + p >= nrows) continue;
        if constexpr (RW == 3) epi.store3((row0 + p) / 3, m, a[m * LS + p], a[m * LS + p + 1], a[m * LS + p + 2]);
        else epi.store2(row0 + p, m, a[m * LS + p], acc);
    }
    if constexpr (NR > 0) {
        __shared__ double red[NR * 16];
        block_sum_any<NR>(acc, red);
        if (threadIdx.x == 0) epi.reduce_out(blockIdx.x, acc);
    }
}

// ------------------------------------------------------ host pass helpers
// Each runs the power-of-two kernel when the length allows it, else the
// any-length kernel.  ``nblocks`` (c2r) receives the workgroup count, which
// indexes the Epi reduction partials.

// Calls f(IC<P>{}) for a shape's pencil count.
template <typename T, class F> inline void with_any_p(const AnyShape& sh, F&& f) {
    constexpr int PM = sizeof(T) == 4 ? 16 : 8;
    if (sh.P == PM) f(IC<PM>{});
    else f(IC<PM / 2>{});
}

inline bool pow2_len(int64_t n, int64_t maxn) { return is_pow2(n) && n >= 4 && n <= maxn; }

template <typename T, int DIR, class Op>
inline int colpass(int64_t n, int64_t planes, int64_t ncols, int64_t plane_stride, int64_t es, const c2<T>* tw, const Op& op,
                   hipStream_t st, const char* tname = "colpass") {
    if (pow2_len(n, 1024)) {
        dispatch_n(n, [&](auto N) {
            const ColGeom g = col_geom<T, decltype(N)::value>(planes, ncols, plane_stride, es);
            launch_colpass<T, decltype(N)::value, DIR>(g, tw, op, st, tname);
        });
        return LDL_OK;
    }
    AnyPlan pl;
    if (!any_plan(n, &pl)) return fail(LDL_EUNSUPPORTED, "FFT length must have no prime factor other than 2, 3 and 5");
    const c2<T>* twn;
    int rc = twiddles_n<T>((int)n, &twn);
    if (rc) return rc;
    const AnyShape sh = any_shape<T>(&pl, (int)n, (int)n, planes * ncols);
    KTimer _t(tname, st);
    with_any_p<T>(sh, [&](auto PC) {
        constexpr int P = decltype(PC)::value;
        ColGeom g{planes, ncols, plane_stride, es, (ncols + P - 1) / P, 0};
        g.ntiles = g.tiles_per_plane * planes;
        allow_lds(&k_colpass_any<T, DIR, P, Op>, sh.lds);
        hipLaunchKernelGGL((k_colpass_any<T, DIR, P, Op>), dim3((unsigned)g.ntiles), dim3(sh.th), sh.lds, st, g, twn, pl, op);
    });
    return LDL_OK;
}

template <typename T, class Pro, class Epi>
inline int zpass_r2c(int64_t nrows, int64_t n2, const c2<T>* tw, const Pro& pro, const Epi& epi, hipStream_t st,
                     const char* tname = "zpass_r2c") {
    if (pow2_len(n2 / 2, 512) && n2 % 2 == 0) {
        dispatch_h(n2 / 2, [&](auto H) { launch_zr2c<T, decltype(H)::value>(nrows, tw, pro, epi, st, tname); });
        return LDL_OK;
    }
    AnyPlan pl;
    if (n2 % 2 || !any_plan(n2 / 2, &pl)) return fail(LDL_EUNSUPPORTED, "FFT last axis must be even with no prime factor other than 2, 3 and 5");
    const c2<T>* tw2;
    int rc = twiddles_n<T>((int)n2, &tw2);
    if (rc) return rc;
    const AnyShape sh = any_shape<T>(&pl, (int)(n2 / 2), (int)n2, nrows);
    KTimer _t(tname, st);
    with_any_p<T>(sh, [&](auto PC) {
        constexpr int P = decltype(PC)::value;
        allow_lds(&k_zpass_r2c_any<T, P, Pro, Epi>, sh.lds);
        hipLaunchKernelGGL((k_zpass_r2c_any<T, P, Pro, Epi>), dim3((unsigned)((nrows + P - 1) / P)), dim3(sh.th), sh.lds, st, nrows, tw2, pl, pro,
                           epi);
    });
    return LDL_OK;
}

// Workgroup count of zpass_c2r over nrows rows of n2 (its reduction partials).
template <typename T>
inline int64_t zpass_c2r_blocks(int64_t nrows, int64_t n2) {
    int64_t nb = 0;
    if (pow2_len(n2 / 2, 512) && n2 % 2 == 0) {
        dispatch_h(n2 / 2, [&](auto H) { nb = (nrows + FftCfg<T, decltype(H)::value>::P - 1) / FftCfg<T, decltype(H)::value>::P; });
    } else {
        AnyPlan pl;
        if (!any_plan(n2 / 2, &pl)) return 0;
        const int P = any_shape<T>(&pl, (int)(n2 / 2), (int)n2, nrows).P;
        nb = (nrows + P - 1) / P;
    }
    return nb;
}

template <typename T, class Pro, class Epi>
inline int zpass_c2r(int64_t nrows, int64_t n2, const c2<T>* tw, const Pro& pro, const Epi& epi, hipStream_t st, int64_t* nblocks,
                     const char* tname = "zpass_c2r") {
    if (pow2_len(n2 / 2, 512) && n2 % 2 == 0) {
        dispatch_h(n2 / 2, [&](auto H) {
            constexpr int HH = decltype(H)::value;
            constexpr int RPB = zc2r_rows_per_block<T, HH, Epi>();
            if (nblocks) *nblocks = (nrows + RPB - 1) / RPB;
            launch_zc2r<T, HH>(nrows, tw, pro, epi, st, tname);
        });
        return LDL_OK;
    }
    AnyPlan pl;
    if (n2 % 2 || !any_plan(n2 / 2, &pl)) return fail(LDL_EUNSUPPORTED, "FFT last axis must be even with no prime factor other than 2, 3 and 5");
    const c2<T>* tw2;
    int rc = twiddles_n<T>((int)n2, &tw2);
    if (rc) return rc;
    const AnyShape sh = any_shape<T>(&pl, (int)(n2 / 2), (int)n2, nrows);
    KTimer _t(tname, st);
    with_any_p<T>(sh, [&](auto PC) {
        constexpr int P = decltype(PC)::value, RPB = any_rows<Epi, P>();
        const int64_t nb = (nrows + RPB - 1) / RPB;
        if (nblocks) *nblocks = nb;
        allow_lds(&k_zpass_c2r_any<T, P, Pro, Epi>, sh.lds);
        hipLaunchKernelGGL((k_zpass_c2r_any<T, P, Pro, Epi>), dim3((unsigned)nb), dim3(sh.th), sh.lds, st, nrows, tw2, pl, pro, epi);
    });
    return LDL_OK;
}

}  // namespace ldl
