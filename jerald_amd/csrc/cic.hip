// CIC paint (particle -> mesh) and readout (mesh -> particle) on gfx950.
//
// Algorithm (lib/parops_fast.h:353-481, :615-821, single rank): x = mesh
// coordinate, i = floor(x) wrapped mod N, f = x - i; corner (i+a, j+b, k+c)
// gets weight w_x[a] w_y[b] w_z[c] with w[0] = 1 - f, w[1] = f.
//
// Paint accumulates in fixed point: each deposit is an integer multiple of
// 2^-s and deposits are summed with integer adds, so the density is
// bit-identical for any particle order or scheduling.  s is chosen per call
// from max|m| and Np so that no cell (nor the total) can overflow.  The
// rounded mass rint(m 2^s) is split over the corners x, then y, then z, each
// split truncating toward zero, so the painted total equals the sum of the
// rounded masses exactly and every deposit has the sign of its mass.
#include "cic.h"

#include <algorithm>
#include <mutex>
#include <vector>

namespace ldl {

// ---------------------------------------------------------- host drivers
static constexpr int kBlock = 256;
static constexpr int64_t kHdrBytes = 256;

// Tiles of the tiled paint: 8 x 16 x 32 cells (z fastest) = 32 KB of 64-bit
// LDS accumulators per component (one component: several workgroups per CU;
// three: 96 KB, one workgroup of 1024 threads per CU).  Long z runs keep the
// particles a tile reads from the lattice-ordered arrays in runs of 32
// consecutive rows' worth of bytes, so fewer cache lines straddle two tiles.
// The 32-bit three-component paint holds 48 KB: three workgroups of 512
// threads per CU (6 waves per SIMD), so one tile's LDS clear and write-out
// overlap the others' deposits.
static constexpr int kTileX = 8, kTileY = 16, kTileZ = 32;
static constexpr int kAcc32Block = 512;
// One component (32 KB of 64-bit accumulators): 512 threads with 4 particles
// each per round, 62 VGPRs, four workgroups per CU (0.84 ms per 512^3 launch
// against 0.91 for 256 threads with 6).
static constexpr int kPaint1Block = 512;

static inline size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }

// Stray lists (cic.h) for absolute positions, whose order is the caller's, from
// 2^22 particles on, and on meshes whose keys fit their bins (1024^3 has 2^21
// keys).  When every particle is in order they cost three nearly empty launches
// and the bins' scan, 7 to 25 us at any size (512^3: sort 0.768 -> 0.795 ms), so
// below the line that is a quarter of the paint and more; out of order they pay
// from 2^20 on, by the more the more particles there are.  FP32 paint, us,
// without -> with lists, in order, 40% in clumps, shuffled: 2^20 particles on
// 128^3 48 -> 66, 115 -> 86, 161 -> 93; 2^22 on 160^3 83 -> 104, 274 -> 193, 386
// -> 239; 2^22 on 320^3 127 -> 142, 352 -> 216, 498 -> 267; 2^24 on 256^3 283 ->
// 290, 1328 -> 615, 2541 -> 844.  Displacements from a lattice are in order by
// construction and sort without.
static constexpr int64_t kStrayMin = 1 << 22;
static constexpr int kSortPPT = 8;  // particles per thread of the sort's passes: chunks of 2048
// Below 2^20 particles (512 chunks of 2048, two per CU) chunks of 512 spread
// the passes over more CUs; key and scatter pass, us: 64^3 9.8 and 8.4 -> 7.5
// and 6.6, 100^3 12.3 and 9.7 -> 10 and 8.8, FP64 14.8 and 9.5 -> 12 and 8.7.
// 128^3 takes 15 and 12 either way, 160^3 the scatter 16.6 -> 18.6.
static constexpr int kFewPPT = 2;
static constexpr int64_t kFew = 1 << 20;
static_assert(kFew <= kStrayMin, "the scatter of few particles places every key, listed ones too");
static inline int64_t sort_chunks(int64_t np) { return (np + 256 * kSortPPT - 1) / (256 * kSortPPT); }
// Workgroups of the key pass with lists: two chunks each or more.
static inline int64_t stray_groups(int64_t np) { return std::max<int64_t>(1, std::min<int64_t>(kSegs, sort_chunks(np) / 2)); }
static inline int64_t stray_group_size(int64_t np) { return (sort_chunks(np) + stray_groups(np) - 1) / stray_groups(np) * 256 * kSortPPT; }

// Which tiles a paint takes.  A sort handed from one paint to another (bins)
// is read with the tiles it was written with: both ask with the same mesh,
// particles and accumulator width.
//
// kSplitSmall: a mesh of fewer large tiles than the card has CUs (256) leaves
// CUs idle, each busy one behind a chain of clear, deposit and write-out;
// 4 x 8 x 16 cells with 256 threads are eight times the workgroups with a
// shorter chain each.  One and three components, us, large tiles -> small: 64^3
// FP32 15 and 22 -> 13 and 14, FP64 20 and 36 -> 14 and 22; 80^3 (150 large
// tiles) 17 and 23 -> 15 and 18, FP64 21 and 37 -> 17 and 29; 100^3 (364) 20
// and 29 -> 21 and 28 with a longer scan; 128^3 (512) 22 and 33 -> 28 and 40.
// From kStrayMin particles on the large tiles stay: the sort's lists and the
// fixed scratch of the paint without allocation are sized with them.
//
// kSplitFlat: 8 x 16 x 16 cells where three components take 64-bit sums (FP64,
// with the one-component paint that hands its sort over, and the FP32
// three-component paint without a density).  48 KB instead of 96 KB hold three workgroups of 512
// threads per CU instead of one of 1024, so that clearing, loading, depositing
// and writing out of different tiles overlap.  256^3, us: FP64 607 -> 496,
// FP32 339 -> 281; FP64 one component (256 threads) 223 -> 205.  The 32-bit
// paints have that occupancy with the longer z runs, and the FP64 one-component
// paint on its own keeps the workspace it had.  Meshes whose keys would
// no longer fit the stray lists (FP64 at 1024^3) keep the large tiles.
//
// A workspace with room for the large tiles' keys alone takes those in place of
// either split.
template <int N> using Int = std::integral_constant<int, N>;
enum Split { kSplitLarge, kSplitSmall, kSplitFlat };
static constexpr int kSmallX = 4, kSmallY = 8, kSmallZ = 16, kSmallBlock = 256;
static constexpr int kFlatZ = 16, kFlat1Block = 256, kFlat3Block = 512;
struct PaintTiles {
    TileGeom tg;
    Split split;
};
static PaintTiles paint_tiles(const Mesh& m, int64_t np, bool wide, bool large_only = false) {
    static const int large[3] = {3, 4, 5}, small[3] = {2, 3, 4}, flats[3] = {3, 4, 4};
    const TileGeom tg = make_tiles(m, large);
    if (large_only) return {tg, kSplitLarge};
    if (tg.ntiles < 256 && np < kStrayMin) return {make_tiles(m, small), kSplitSmall};
    if (!wide) return {tg, kSplitLarge};
    const TileGeom tf = make_tiles(m, flats);
    if (tf.nkeys() > ((int64_t)kBins << kBinKeysLog)) return {tg, kSplitLarge};
    return {tf, kSplitFlat};
}

// Workspace: header | direct-mode mesh (nc, LDL_PAINT_DIRECT only) | counts
// and the strays' bins | offsets | segment sums | key | sorted | stray lists
struct PaintWs {
    size_t acc, counts, bins, offsets, segsum, key, sorted, list, pair, seg, off, total;
    bool strays;
};
static bool paint_direct(int32_t flags) { return (flags & LDL_PAINT_DIRECT) && !(flags & LDL_PAINT_FLOAT_ATOMIC); }
static PaintWs paint_ws(const Mesh& m, int nc, int64_t np, int32_t flags, const TileGeom& tg, bool lists) {
    const int64_t nk = tg.nkeys();
    PaintWs w;
    w.acc = al256((size_t)kHdrBytes);
    w.counts = w.acc + (paint_direct(flags) ? al256((size_t)nc * m.cells() * 8) : 0);
    w.strays = lists && !paint_direct(flags) && np >= kStrayMin && nk <= ((int64_t)kBins << kBinKeysLog);
    w.bins = w.counts + (size_t)nk * 4;  // cleared together
    w.offsets = w.counts + al256((size_t)(nk + 1 + (w.strays ? kBins : 0)) * 4);
    w.segsum = w.offsets + al256((size_t)(nk + 1) * 4);
    w.key = w.segsum + al256((size_t)(nk / kScanSeg + 1) * 4);
    w.sorted = w.key + al256((size_t)np * 4);
    w.list = w.sorted + al256((size_t)np * 4);
    w.pair = w.list + (w.strays ? al256((size_t)(stray_groups(np) * stray_group_size(np)) * 4) : 0);
    w.seg = w.pair + (w.strays ? al256((size_t)np * 8) : 0);
    w.off = w.seg + (w.strays ? al256((size_t)kSegs * 4) : 0);
    w.total = w.off + (w.strays ? (size_t)kSegs * kBins * 4 : 0);
    return w;
}

size_t paint_ws_bytes(const Mesh& m, int nc, int64_t np, int32_t flags) {
    if (flags & LDL_PAINT_FLOAT_ATOMIC) return 0;  // float atomics deposit straight into the output
    np = np < 0 ? 0 : np;
    return paint_ws(m, nc, np, flags, paint_tiles(m, np, nc == 3).tg, !(flags & LDL_PAINT_LATTICE)).total;
}

size_t paint_bins_bytes(const Mesh& m, int64_t np) {
    np = np < 0 ? 0 : np;
    return (size_t)(paint_tiles(m, np, true).tg.nkeys() + 1 + np + 1) * 4;
}

template <typename T>
int paint_impl(const T* pos, const ldl_pos_desc* pdesc, int64_t np, const T* mass, double mscalar, int nc,
               const int64_t nmesh[3], double out_scale, int32_t flags, T* out, void* ws, size_t ws_bytes,
               hipStream_t st, unsigned* bins_out, const unsigned* bins_in, const T* wmesh, double wscale,
               unsigned long long* absmax_in, bool absmax_reset, const AxisTabs<T>& tabs) {
    Mesh m;
    int rc = check_mesh(nmesh, &m);
    if (rc) return rc;
    if (np < 0) return fail(LDL_EINVAL, "np must be >= 0");
    if (!out) return fail(LDL_EINVAL, "out is NULL");
    if (np > 0 && !pos) return fail(LDL_EINVAL, "pos is NULL");
    if (nc == 3 && !mass && np > 0) return fail(LDL_EINVAL, "ppaint3D needs a (Np,3) mass array");
    PosDec<T> pd;
    if ((rc = make_posdec<T>(pdesc, nmesh, np, &pd))) return rc;
    const int64_t cells = m.cells();
    const int64_t tot = (int64_t)nc * cells;
    const unsigned gp = grid_for(np, kBlock, 1 << 16);
    const unsigned gm = grid_for(tot, kBlock, 1 << 16);
    const int mode = flags & 1;
    auto prep = [&](const PaintPrep& a) {
        const int64_t n = std::max<int64_t>(std::max<int64_t>(a.ncounts, tabs.total()), 1);
        hipLaunchKernelGGL(k_paint_prep<T>, dim3(grid_for(n, kBlock, 1 << 12)), dim3(kBlock), 0, st, a, tabs);
    };
    if (mode == LDL_PAINT_FLOAT_ATOMIC) {
        if (tabs.total() || (absmax_in && absmax_reset))
            prep(PaintPrep{nullptr, 0, absmax_reset ? absmax_in : nullptr, nc, 1, nullptr, 0.0, nullptr, nullptr, 0});
        hipLaunchKernelGGL(k_fill<T>, dim3(gm), dim3(kBlock), 0, st, out, tot, T(0));
        if (np > 0) {
            if (nc == 1)
                { KTimer _t("paint_deposit", st); hipLaunchKernelGGL((k_paint_float<T, 1>), dim3(gp), dim3(kBlock), 0, st, pos, pd, np, mass, (T)mscalar, (T)out_scale, m, out); }
            else
                { KTimer _t("paint_deposit", st); hipLaunchKernelGGL((k_paint_float<T, 3>), dim3(gp), dim3(kBlock), 0, st, pos, pd, np, mass, (T)mscalar, (T)out_scale, m, out); }
        }
        LDL_LAUNCH_CHECK();
        return LDL_OK;
    }
    if (np > (int64_t)0xFFFFFFFFll) return fail(LDL_EUNSUPPORTED, "paint supports np < 2^32");
    // a workspace without room for the stray lists (ldl_ppaint_noalloc's fixed
    // one, or one sized for lattice positions) or the smaller tiles' keys sorts
    // without them
    const bool wide = sizeof(T) == 8 ? nc == 3 || bins_in || bins_out : nc == 3 && !wmesh;
    PaintTiles pt = paint_tiles(m, np, wide);
    PaintWs w = paint_ws(m, nc, np, flags, pt.tg, pd.physical());
    if (ws && ws_bytes < w.total) w = paint_ws(m, nc, np, flags, pt.tg, false);
    if (ws && ws_bytes < w.total && !bins_in && !bins_out) {
        pt = paint_tiles(m, np, wide, true);
        w = paint_ws(m, nc, np, flags, pt.tg, false);
    }
    if (!ws || ws_bytes < w.total) return fail(LDL_EINVAL, "paint workspace too small (see ldl_paint_workspace_bytes)");
    char* wb = reinterpret_cast<char*>(ws);
    auto* hdr = reinterpret_cast<unsigned long long*>(wb);
    auto* acc = reinterpret_cast<unsigned long long*>(wb + w.acc);
    // header: max |m| bits; for a scalar mass it is known on the host
    unsigned long long hbits = 0;
    if (!mass) {
        double a = std::fabs((double)(T)mscalar);
        std::memcpy(&hbits, &a, 8);
    }
    static_assert(kHdrSlots * 8 == kHdrBytes, "the header's slots fill it");
    if (!mass) absmax_in = nullptr;  // max |m| per component may be handed over by the kernel that wrote the masses
    PaintPrep pp{hdr, hbits, absmax_in, nc, absmax_reset, nullptr, 0.0, nullptr, nullptr, 0};
    auto absmax = [&]() {
        if (!mass || absmax_in || np == 0) return;
        KTimer _t("paint_absmax", st);
        // two workgroups per CU keep 8 MB of loads in flight; more of them, all
        // ending at once, only queue on the maximum's address (3.4e6 FP64
        // masses: 51 us with 4096 workgroups, 8 with 512)
        const dim3 ga(grid_for((np * nc * (int64_t)sizeof(T) + 63) / 64, kBlock, 512));
        if (nc == 1) hipLaunchKernelGGL((k_absmax<T, 1>), ga, dim3(kBlock), 0, st, mass, np, hdr);
        else hipLaunchKernelGGL((k_absmax<T, 3>), ga, dim3(kBlock), 0, st, mass, np, hdr);
    };
    if (flags & LDL_PAINT_DIRECT) {
        prep(pp);
        absmax();
        // reference variant: one device-scope 64-bit atomic per corner
        if (!(flags & LDL_PAINT_WS_ZEROED))
            hipLaunchKernelGGL(k_fill_u64, dim3(gm), dim3(kBlock), 0, st, acc, tot, 0ull);
        if (np > 0) {
            if (nc == 1)
                { KTimer _t("paint_deposit", st); hipLaunchKernelGGL((k_paint_fixed<T, 1>), dim3(gp), dim3(kBlock), 0, st, pos, pd, np, mass, (T)mscalar, m, acc, hdr); }
            else
                { KTimer _t("paint_deposit", st); hipLaunchKernelGGL((k_paint_fixed<T, 3>), dim3(gp), dim3(kBlock), 0, st, pos, pd, np, mass, (T)mscalar, m, acc, hdr); }
        }
        if (nc == 1)
            { KTimer _t("paint_convert", st); hipLaunchKernelGGL((k_fixed_to_float<T, 1>), dim3(grid_for(cells, kBlock, 1 << 16)), dim3(kBlock), 0, st, acc, hdr, np, cells, out_scale, out); }
        else
            { KTimer _t("paint_convert", st); hipLaunchKernelGGL((k_fixed_to_float<T, 3>), dim3(grid_for(cells, kBlock, 1 << 16)), dim3(kBlock), 0, st, acc, hdr, np, cells, out_scale, out); }
        LDL_LAUNCH_CHECK();
        return LDL_OK;
    }
    // tiled path: counting sort by (tile, face class), then one workgroup per
    // tile sums the tile's cells completely in LDS.  A 3-component paint that
    // is handed the sort of an earlier 1-component paint of the same positions
    // (bins_in) skips the sort.
    const TileGeom& tg = pt.tg;
    const int64_t nk = tg.nkeys();
    if (m.n0 >= (1ll << 31) || m.n1 >= (1ll << 31) || m.n2 >= (1ll << 31) || nk >= (1ll << 32))
        return fail(LDL_EUNSUPPORTED, "the tiled paint takes mesh axes below 2^31 cells and fewer than 2^29 tiles");
    // (the sort and deposit kernels must use the same decode)
    const int dm = decode_mode(pd, mesh_pow2(m));
    auto with_dm = [dm](auto&& f) {
        switch (dm) {
            case kDecLU: f(std::integral_constant<int, kDecLU>{}); break;
            case kDecP2: f(std::integral_constant<int, kDecP2>{}); break;
            case kDecPhysP2: f(std::integral_constant<int, kDecPhysP2>{}); break;
            case kDecPhys: f(std::integral_constant<int, kDecPhys>{}); break;
            default: f(std::integral_constant<int, kDecAny>{}); break;
        }
    };
    const MeshP2 mp = mesh_p2(m);
    auto* counts = reinterpret_cast<unsigned*>(wb + w.counts);
    auto* segsum = reinterpret_cast<unsigned*>(wb + w.segsum);
    auto* key = reinterpret_cast<unsigned*>(wb + w.key);
    unsigned* offsets = reinterpret_cast<unsigned*>(wb + w.offsets);
    unsigned* sorted = reinterpret_cast<unsigned*>(wb + w.sorted);
    // the FP32 1-component paint that hands its sort over also records its
    // largest cell there; a 3-component paint handed that sort reads it in place
    // of scanning the density
    unsigned* vmax_out = nullptr;
    if (bins_out) {
        offsets = bins_out;
        sorted = bins_out + nk + 1;
        if (nc == 1 && sizeof(T) == 4) vmax_out = bins_out + nk + 1 + np;
    }
    pp.vmax_out = vmax_out;
    if (!bins_in) {
        pp.counts = counts;
        pp.ncounts = nk + (w.strays ? kBins : 0);
    } else if (nc == 3 && sizeof(T) == 4 && wmesh) {
        // recorded by the 1-component paint that wrote the sort and wmesh
        pp.vmax_in = bins_in + nk + 1 + np;
        pp.wscale = wscale;
    }
    prep(pp);
    absmax();
    if (bins_in) {
        offsets = const_cast<unsigned*>(bins_in);
        sorted = const_cast<unsigned*>(bins_in) + nk + 1;
    } else {
        const bool few = np < kFew;
        const int64_t nchunks = few ? (np + 256 * kFewPPT - 1) / (256 * kFewPPT) : sort_chunks(np);
        StrayLists sl{};
        if (w.strays) {
            auto u = [&](size_t off) { return reinterpret_cast<unsigned*>(wb + off); };
            sl = StrayLists{u(w.list), reinterpret_cast<uint2*>(wb + w.pair), u(w.seg), u(w.off), u(w.bins), stray_group_size(np), 0};
            while (((int64_t)kBins << sl.shift) < nk) sl.shift++;
        }
        const dim3 gb(w.strays ? (unsigned)stray_groups(np) : grid_for(nchunks, 1, 1 << 15));
        if (np > 0) {
            KTimer _t("paint_bin", st);
            with_dm([&](auto D) {
                constexpr int DM = decltype(D)::value;
                if constexpr (DM == kDecPhysP2 || DM == kDecPhys) {
                    if (w.strays) {
                        hipLaunchKernelGGL((k_bin_keys<T, kSortPPT, DM, true>), gb, dim3(256), 0, st, pos, pd, np, mp, tg, counts, key, sl);
                        return;
                    }
                }
                if (few) hipLaunchKernelGGL((k_bin_keys<T, kFewPPT, DM, false>), gb, dim3(256), 0, st, pos, pd, np, mp, tg, counts, key, sl);
                else hipLaunchKernelGGL((k_bin_keys<T, kSortPPT, DM, false>), gb, dim3(256), 0, st, pos, pd, np, mp, tg, counts, key, sl);
            });
            if (w.strays) {
                hipLaunchKernelGGL(k_stray_part, gb, dim3(kStrayThreads), 0, st, key, sl);
                hipLaunchKernelGGL(k_stray_count, dim3(1024), dim3(kStrayThreads), 0, st, sl, counts);
            }
        }
        {
            KTimer _t("paint_scan", st);
            const unsigned nseg = (unsigned)((nk + kScanSeg - 1) / kScanSeg);
            if (nseg > 1) hipLaunchKernelGGL(k_scan_sums, dim3(nseg), dim3(1024), 0, st, counts, nk, segsum);
            hipLaunchKernelGGL(k_scan_apply, dim3(nseg), dim3(1024), 0, st, counts, nk, segsum, offsets, counts);  // counts become the cursors
        }
        if (np > 0) {
            KTimer _t("paint_scatter", st);
            const dim3 gs(grid_for(nchunks, 1, 1 << 15));
            if (few) hipLaunchKernelGGL(k_bin_scatter<kFewPPT>, gs, dim3(256), 0, st, np, key, 0u, counts, sorted);
            else hipLaunchKernelGGL(k_bin_scatter<kSortPPT>, gs, dim3(256), 0, st, np, key, w.strays ? kStrayBit : 0u, counts, sorted);
            if (w.strays) hipLaunchKernelGGL(k_stray_scatter, dim3(1024), dim3(kStrayThreads), 0, st, sl, counts, sorted);
        }
    }
    if (nc == 3 && sizeof(T) == 4 && wmesh && !bins_in) {
        KTimer _t("paint_absmax", st);
        hipLaunchKernelGGL(k_mesh_absmax<T>, dim3(grid_for(cells, kBlock, 512)), dim3(kBlock), 0, st, wmesh, cells, wscale, hdr + 3);
    }
    // one workgroup of TB threads per tile of TX x TY x TZ cells; ACC32: FP32
    // with the positions' unit-mass density known takes 32-bit accumulators
    auto deposit = [&](auto NC, auto TX, auto TY, auto TZ, auto TB, auto ACC32) {
        constexpr int nc_ = decltype(NC)::value, tb = decltype(TB)::value;
        with_dm([&](auto D) {
            hipLaunchKernelGGL((k_paint_tiles<T, nc_, decltype(TX)::value, decltype(TY)::value, decltype(TZ)::value, tb, decltype(D)::value,
                                              decltype(ACC32)::value != 0>),
                               dim3((unsigned)tg.ntiles), dim3(tb), 0, st, pos, pd, np, mass, (T)mscalar, m, mp, tg, offsets, sorted, hdr, out_scale, out,
                               nc_ == 1 ? vmax_out : nullptr);
        });
    };
    KTimer _t(nc == 1 ? "paint_deposit1" : "paint_deposit3", st);
    constexpr Int<0> no{};
    constexpr Int<1> c1{};
    constexpr Int<3> c3{};
    const bool acc32 = sizeof(T) == 4 && nc == 3 && wmesh;
    auto small = [&](auto NC, auto ACC32) { deposit(NC, Int<kSmallX>{}, Int<kSmallY>{}, Int<kSmallZ>{}, Int<kSmallBlock>{}, ACC32); };
    auto flat = [&](auto NC, auto TB) { deposit(NC, Int<kTileX>{}, Int<kTileY>{}, Int<kFlatZ>{}, TB, no); };
    auto large = [&](auto NC, auto TB, auto ACC32) { deposit(NC, Int<kTileX>{}, Int<kTileY>{}, Int<kTileZ>{}, TB, ACC32); };
    if (acc32) {
        if constexpr (sizeof(T) == 4) {
            if (pt.split == kSplitSmall) small(c3, c1);
            else large(c3, Int<kAcc32Block>{}, c1);
        }
    } else if (pt.split == kSplitSmall) {
        if (nc == 1) small(c1, no);
        else small(c3, no);
    } else if (pt.split == kSplitFlat) {
        if (nc == 3) flat(c3, Int<kFlat3Block>{});
        else if constexpr (sizeof(T) == 8) flat(c1, Int<kFlat1Block>{});
    } else if (nc == 1) {
        large(c1, Int<kPaint1Block>{}, no);
    } else {
        large(c3, Int<1024>{}, no);
    }
    LDL_LAUNCH_CHECK();
    return LDL_OK;
}

template <typename T>
int readout_impl(const T* pos, const ldl_pos_desc* pdesc, int64_t np, const T* field, const int64_t nmesh[3],
                 int kind, int vjpdim, const T* aux, T* out, hipStream_t st) {
    Mesh m;
    int rc = check_mesh(nmesh, &m);
    if (rc) return rc;
    if (np < 0) return fail(LDL_EINVAL, "np must be >= 0");
    if (np == 0) return LDL_OK;
    if (!pos || !field || !out) return fail(LDL_EINVAL, "NULL array argument");
    PosDec<T> pd;
    if ((rc = make_posdec<T>(pdesc, nmesh, np, &pd))) return rc;
    const Sweep sw = make_sweep(pd, np);
    const unsigned g = sweep_grid(sw);
    static_assert(kBlock == kChunk, "gathers take one particle per thread");
    if (kind == 0 && (vjpdim < -1 || vjpdim > 2)) return fail(LDL_EINVAL, "vjpdim must be between -1 and 2");
    if (kind == 3 && !aux) return fail(LDL_EINVAL, "v3 is NULL");
    KTimer _t("readout", st);
    switch (kind) {
        case 0:
            with_geom<T>(m, pd, [&](auto geo) {
                hipLaunchKernelGGL((k_readout<T, decltype(geo)>), dim3(g), dim3(kBlock), 0, st, pos, pd, np, sw, field, geo, vjpdim, out);
            });
            break;
        case 1:
            with_geom<T>(m, pd, [&](auto geo) {
                hipLaunchKernelGGL((k_readout3<T, decltype(geo)>), dim3(g), dim3(kBlock), 0, st, pos, pd, np, sw, fields3(field, m.cells()), geo, out);
            });
            break;
        case 2:
            with_geom<T>(m, pd, [&](auto geo) {
                hipLaunchKernelGGL((k_readout_grad<T, decltype(geo)>), dim3(g), dim3(kBlock), 0, st, pos, pd, np, sw, field, geo, aux, out);
            });
            break;
        case 3:
            with_geom<T>(m, pd, [&](auto geo) {
                hipLaunchKernelGGL((k_readout_grad3<T, decltype(geo)>), dim3(g), dim3(kBlock), 0, st, pos, pd, np, sw, fields3(field, m.cells()), aux, geo, out);
            });
            break;
    }
    LDL_LAUNCH_CHECK();
    return LDL_OK;
}

template int paint_impl<float>(const float*, const ldl_pos_desc*, int64_t, const float*, double, int, const int64_t*, double, int32_t, float*, void*,
                               size_t, hipStream_t, unsigned*, const unsigned*, const float*, double, unsigned long long*, bool, const AxisTabs<float>&);
template int paint_impl<double>(const double*, const ldl_pos_desc*, int64_t, const double*, double, int, const int64_t*, double, int32_t, double*,
                                void*, size_t, hipStream_t, unsigned*, const unsigned*, const double*, double, unsigned long long*, bool, const AxisTabs<double>&);
template int readout_impl<float>(const float*, const ldl_pos_desc*, int64_t, const float*, const int64_t*, int, int, const float*, float*, hipStream_t);
template int readout_impl<double>(const double*, const ldl_pos_desc*, int64_t, const double*, const int64_t*, int, int, const double*, double*, hipStream_t);

// ------------------------------------------------ allocation-free paint
// ldl_ppaint_noalloc_* paint with this fixed device array as their workspace,
// for callers that cannot allocate (graph capture, serving loops).  Host code
// reaches it only through the address hipGetSymbolAddress returns for the
// current device (the array's name is a host-side stand-in there); every
// call on a device shares that device's copy.
static constexpr size_t kNoAllocScratchBytes = (size_t)64 << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

static std::mutex g_scratch_mutex;
static std::vector<void*> g_scratch_ptr;  // per device id

static int noalloc_scratch(void** out) {
    int dev = 0;
    LDL_HIP_TRY(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if ((int)g_scratch_ptr.size() <= dev) g_scratch_ptr.resize(dev + 1, nullptr);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(LDL_EHIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return LDL_OK;
}

template <typename T>
static int paint_noalloc(const T* pos, const ldl_pos_desc* pdesc, int64_t np, const T* mass, double mscalar, const int64_t nmesh[3],
                         double out_scale, int32_t flags, T* out, hipStream_t st) {
    Mesh m;
    int rc = check_mesh(nmesh, &m);
    if (rc) return rc;
    if (np < 0) return fail(LDL_EINVAL, "np must be >= 0");
    // the array holds whatever the previous call left: never skip clearing
    flags &= ~LDL_PAINT_WS_ZEROED;
    const size_t need = flags & LDL_PAINT_FLOAT_ATOMIC ? 0 : paint_ws(m, 1, np, flags, paint_tiles(m, np, false).tg, false).total;  // (sorts without the stray lists)
    if (need > kNoAllocScratchBytes)
        return fail(LDL_EINVAL, "ldl_ppaint_noalloc: this paint needs " + std::to_string(need) + " bytes of scratch, the fixed array holds " +
                                    std::to_string(kNoAllocScratchBytes) + " (use ldl_ppaint with a workspace)");
    void* ws = nullptr;
    if ((rc = noalloc_scratch(&ws))) return rc;
    return paint_impl<T>(pos, pdesc, np, mass, mscalar, 1, nmesh, out_scale, flags, out, ws, kNoAllocScratchBytes, st);
}

}  // namespace ldl

using namespace ldl;

extern "C" {

int ldl_ppaint_noalloc_f32(const float* pos, const ldl_pos_desc* pd, int64_t np, const float* mass, double mass_scalar,
                           const int64_t nmesh[3], double out_scale, int32_t flags, float* out, void* stream) {
    return paint_noalloc<float>(pos, pd, np, mass, mass_scalar, nmesh, out_scale, flags, out, as_stream(stream));
}
int ldl_ppaint_noalloc_f64(const double* pos, const ldl_pos_desc* pd, int64_t np, const double* mass, double mass_scalar,
                           const int64_t nmesh[3], double out_scale, int32_t flags, double* out, void* stream) {
    return paint_noalloc<double>(pos, pd, np, mass, mass_scalar, nmesh, out_scale, flags, out, as_stream(stream));
}

size_t ldl_paint_workspace_bytes(const int64_t nmesh[3], int32_t ncomp, int64_t np, int32_t flags) {
    Mesh m;
    if (check_mesh(nmesh, &m) || (ncomp != 1 && ncomp != 3) || np < 0) return 0;
    return paint_ws_bytes(m, ncomp, np, flags);
}

#define PAINT_ENTRY(SUF, T)                                                                                      \
    int ldl_ppaint_##SUF(const T* pos, const ldl_pos_desc* pd, int64_t np, const T* mass, double mass_scalar,    \
                         const int64_t nmesh[3], double out_scale, int32_t flags, T* out, void* ws, size_t wsb,  \
                         void* stream) {                                                                        \
        return paint_impl<T>(pos, pd, np, mass, mass_scalar, 1, nmesh, out_scale, flags, out, ws, wsb, as_stream(stream)); \
    }                                                                                                            \
    int ldl_ppaint3D_##SUF(const T* pos, const ldl_pos_desc* pd, int64_t np, const T* mass3, const int64_t nmesh[3], \
                           double out_scale, int32_t flags, T* out, void* ws, size_t wsb, void* stream) {        \
        return paint_impl<T>(pos, pd, np, mass3, 0.0, 3, nmesh, out_scale, flags, out, ws, wsb, as_stream(stream)); \
    }                                                                                                            \
    int ldl_preadout_##SUF(const T* pos, const ldl_pos_desc* pd, int64_t np, const T* field, const int64_t nmesh[3], \
                           int32_t vjpdim, T* out, void* stream) {                                               \
        return readout_impl<T>(pos, pd, np, field, nmesh, 0, vjpdim, nullptr, out, as_stream(stream));          \
    }                                                                                                            \
    int ldl_preadout3D_##SUF(const T* pos, const ldl_pos_desc* pd, int64_t np, const T* field,                  \
                             const int64_t nmesh[3], int32_t vjp, const T* pscale, T* out, void* stream) {       \
        if (!vjp && pscale) return fail(LDL_EINVAL, "pscale is only defined for vjp != 0");                     \
        return readout_impl<T>(pos, pd, np, field, nmesh, vjp ? 2 : 1, -1, pscale, out, as_stream(stream));     \
    }                                                                                                            \
    int ldl_readout_grad3_##SUF(const T* pos, const ldl_pos_desc* pd, int64_t np, const T* fields3, const T* v3, \
                                const int64_t nmesh[3], T* out, void* stream) {                                  \
        return readout_impl<T>(pos, pd, np, fields3, nmesh, 3, -1, v3, out, as_stream(stream));                 \
    }

PAINT_ENTRY(f32, float)
PAINT_ENTRY(f64, double)

}  // extern "C"
