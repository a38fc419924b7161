// Host side of the MFMA GEMM: tile configuration per type and dispatch over the transpose layouts.
// The kernel templates and their design notes are in gemm_kernel.h (every shape and type); hgemm_launch.h and
// sgemm_launch.h hold the FP16 and FP32 products on direct global→LDS loads.
#include "gemm_kernel.h"
#include <stdlib.h>
#include <string.h>
#include <algorithm>

namespace g9 {

// ---------------- host side ----------------
// Tile configurations, per element type and layout, from a sweep on MI355X at n = 4096 (every variant checked against
// a float64 reference). Big: the steady-state configuration. Small: smaller tiles for products whose big tiles
// would leave most of the 256 CUs idle.
// FP64 products come here. By default the FP16 ones that do are those with odd strides or unaligned operands and those of
// at most a k-step of 64, the FP32 ones those of at most a k-step of 32 and short-K NT products and triangles, in both types
// also rows too far apart for the direct kernels' 32-bit offsets; the rates below are of larger products, as
// GEN9BLAS_HGEMM / GEN9BLAS_SGEMM=generic and a forced split send them here.
//   FP16 256×256, 8 waves (4×2): NN 794, NT 950 TFLOP/s. FP64 256×128, 8 waves (4×2): 70.6 TFLOP/s.
//   FP32 with A k-contiguous: small tiles with 4 waves, many workgroups per CU. NN 64×128: 123 TFLOP/s at n = 4096,
//   117 at n = 2048 (256×128: 117 / 105; 128×128, 64×64, 128×64, 64×256 and 2- or 8-wave variants: 74-118). NT
//   64×64: 126 at n = 4096, 119 on the odd shape 3000×11008×4096 (128×128: 128 / 97, the odd shape's 2064 tiles
//   being four rounds of 512 workgroups and a nearly empty fifth). Transposed A: TN 128×128 125 (256×128: 117),
//   TT 128×64 120 (256×128: 117).
//   Small at n = 1024 (NN): FP32 64×64 (256 tiles, no split) 69 TFLOP/s against 62 for 128×128 split four ways;
//   FP64 64×128 split two ways 43, 64×64 41. Both are beaten by 64×64 tiles with two k groups (launch_layout).
struct TileCfg { int BM, BN, WM, WN; };
// Transposed A, whose staging needs more registers than a wave has at 2 waves per SIMD, keeps FP16 at 4 waves (512
// registers per wave), which still spills 68 (B k-contiguous: 144) bytes per lane.
template <class T, bool AK, bool BKC> struct Cfg;
// small_div: the small tile is taken when the big tiles times small_div are fewer than the CUs.
template <bool AK, bool BKC> struct Cfg<f16, AK, BKC> {
    static constexpr TileCfg big = AK ? TileCfg{256, 256, 4, 2} : TileCfg{256, 256, 2, 2};
    static constexpr TileCfg small{128, 128, 2, 2};
    static constexpr int small_div = 2;
};
template <bool AK, bool BKC> struct Cfg<float, AK, BKC> {
    static constexpr TileCfg big = !AK ? (BKC ? TileCfg{128, 64, 2, 2} : TileCfg{128, 128, 2, 2})
                                       : (BKC ? TileCfg{64, 64, 2, 2} : TileCfg{64, 128, 2, 2});
    static constexpr TileCfg small{64, 64, 2, 2};
    static constexpr int small_div = 1;
};
template <bool AK, bool BKC> struct Cfg<double, AK, BKC> {
    static constexpr TileCfg big{256, 128, 4, 2}, small{64, 128, 2, 2};
    static constexpr int small_div = 2;
};

// GEN9BLAS_SPLITK=n forces n split-K slices (0 or 1: none) and turns the tiles with k groups, the triangle's slices and the
// direct FP32 kernel off, so that the FP32 / FP64 summation order depends on K alone and not on the other sizes; -1 when
// unset.
static int splitk_forced() {
    static int forced = -2;
    if (forced == -2) {
        const char *e = getenv("GEN9BLAS_SPLITK");
        forced = e ? std::max(atoi(e), 0) : -1;
    }
    return forced;
}

// Split-K slices for a single product of `tiles` tiles: doubled while the slices still leave at most one workgroup
// per CU and each slice keeps at least 4 k-steps, up to 8. Without a forced split, s > 1 implies tiles · s ≤ CUs here; the
// direct kernels split further (choose() in hgemm_launch.h and sgemm_launch.h, by the bytes of the slices).
// Splitting changes only the FP32 (FP64) summation order: each slice sums its k-range, the slices are then added in
// order, and alpha/beta and the rounding to the element type are applied once.
static int splitk_slices(long long tiles, int K, int BK, int count) {
    const int forced = splitk_forced();
    if (count != 1) return 1;
    if (forced >= 0) return forced < 1 ? 1 : forced > 64 ? 64 : forced;
    int s = 1;
    while (s < 8 && tiles * s * 2 <= num_cus && K / (s * 2) >= 4 * BK) s *= 2;
    return s;
}

// Tiles for operands that the unchecked loads do not take, or not with 32-bit offsets.
constexpr TileCfg TILE64{64, 64, 2, 2};
// Operands whose rows under a tile of the chosen size span 4 GiB or more take 64×64 tiles with 64-bit offsets.
template <class T, TileCfg C, bool AK, bool BKC> static bool narrow(const GemmParams<typename Mma<T>::Sum> &p) {
    return narrow_ok<T>(AK, p.lda, C.BM, p.M) && narrow_ok<T>(BKC, p.ldb, C.BN, p.N);
}

template <class T, TileCfg C, bool AK, bool BKC, int KG = 1, Loads LOADS = UNCHECKED>
static int launch_t(GemmParams<typename Mma<T>::Sum> p, int count) {
    using S = typename Mma<T>::Sum;
    if constexpr (LOADS == UNCHECKED)
        if (!narrow<T, C, AK, BKC>(p)) return launch_t<T, TILE64, AK, BKC, 1, WIDE>(p, count);
    constexpr int BK = 128 / (int)sizeof(T);
    p.tiles_m = (p.M + C.BM - 1) / C.BM;
    p.tiles_n = (p.N + C.BN - 1) / C.BN;
    if ((long long)p.tiles_m * p.tiles_n > 0x7fffffffLL || count > 65535)
        G9_FAIL(GEN9BLAS_ERR_UNSUPPORTED, "gemm grid too large (%d × %d tiles, batch %d)", p.tiles_m, p.tiles_n, count);
    const long long tiles = (long long)p.tiles_m * p.tiles_n;
    const int split = KG > 1 ? 1 : splitk_slices(tiles, p.K, BK, count);
    const dim3 block(C.WM * C.WN * 64 * KG);
    if (split > 1) {
        static_assert((size_t)C.BM * C.BN * sizeof(S) <= SPLITK_TILE_BYTES_MAX, "split tile beyond the work-space bound");
        p.kper = ((p.K + split - 1) / split + BK - 1) / BK * BK;
        const int ns = (p.K + p.kper - 1) / p.kper;
        void *P;
        G9_TRY(scratch(SLOT_P, (size_t)ns * p.M * p.N * sizeof(S), &P));
        p.P = reinterpret_cast<S *>(P);
        hipLaunchKernelGGL((gemm_kernel<T, C.BM, C.BN, C.WM, C.WN, AK, BKC, true, 0, 0, 1, LOADS>),
                           dim3((unsigned)tiles, (unsigned)ns), block, 0, stream, p);
        G9_HIP(hipGetLastError());
        const long long mn = (long long)p.M * p.N;
        const bool v4 = p.N % 4 == 0;
        const long long work = v4 ? mn / 4 : mn;
        const unsigned blocks = (unsigned)std::min<long long>((work + 255) / 256, (long long)num_cus * 8);
        T *Cp = reinterpret_cast<T *>(p.C);
        if (v4) hipLaunchKernelGGL((splitk_reduce<T, S, true>), dim3(blocks), dim3(256), 0, stream, p.P, Cp, p.ldc, p.M, p.N, ns, p.alpha, p.beta);
        else hipLaunchKernelGGL((splitk_reduce<T, S, false>), dim3(blocks), dim3(256), 0, stream, p.P, Cp, p.ldc, p.M, p.N, ns, p.alpha, p.beta);
        G9_HIP(hipGetLastError());
        return 0;
    }
    const dim3 grid((unsigned)tiles, (unsigned)count);
    hipLaunchKernelGGL((gemm_kernel<T, C.BM, C.BN, C.WM, C.WN, AK, BKC, false, 0, 0, KG, LOADS>), grid, block, 0, stream, p);
    G9_HIP(hipGetLastError());
    return 0;
}

// FP64 products of few tiles: 32×32 tiles, four k groups of one wave each (73 KiB of LDS, two workgroups per CU), or eight
// (which spill 36 bytes per lane) for single products of at most a tile per CU, which split K up to 8 ways before: as many partial sums keep the error
// where it was (500×500×512 against 80-bit sums: split K 2.8e-16, four groups 3.8e-16). A
// wave of a 64×128 or 64×64 tile does 4 to 8 times the MFMAs one after the other while most CUs idle; four k groups hide
// each other's barrier and load waits, and no second pass adds slices of K.
// MI355X, µs, the tiles below (two k groups or split K) -> 32×32 (8 groups): 128³ × 7 13.5 -> 5.9 (6.5), 256³ × 3 22.6 ->
// 7.3 (8.0), 512³ 20.4 -> 10.7 (11.1), 976×500×1024 40.1 -> 26.5 (32.5), 128×4096×128 8.8 -> 7.5, 137×1500×700 23.8 -> 14.6.
// Beyond two workgroups per CU it loses (700×900×300 16.1 against 20.3, 1024³ 44 against 48), and so it does to split K
// where that applies (fewer than CUs / 2 tiles of 64×64) with many k-steps: 500×500×5000 57 against 67, 200×200×4000 44
// against 54; the lines of both cross between K = 1600 and 3500.
static long long tiles32(int M, int N, int count) { return (long long)((M + 31) / 32) * ((N + 31) / 32) * count; }
constexpr TileCfg TILE32{32, 32, 1, 1};
constexpr int TILE32_SPLIT_K = 1536;

template <class T, bool AK, bool BKC>
static int launch_layout(const GemmParams<typename Mma<T>::Sum> &p, int count) {
    using CF = Cfg<T, AK, BKC>;
    if constexpr (sizeof(T) < 8 && !(AK && BKC))
        if (!unchecked_ok<T>(AK, p.lda) || !unchecked_ok<T>(BKC, p.ldb)) return launch_t<T, TILE64, AK, BKC, 1, CHECKED>(p, count);
    if constexpr (sizeof(T) == 8) {
        const long long t64 = (long long)((p.M + 63) / 64) * ((p.N + 63) / 64) * count;
        const long long t32 = tiles32(p.M, p.N, count);
        if (splitk_forced() < 0 && t32 <= 2LL * num_cus && (count > 1 || t64 * 2 >= num_cus || p.K <= TILE32_SPLIT_K))
            return count == 1 && t32 <= num_cus ? launch_t<T, TILE32, AK, BKC, 8>(p, count)
                                                : launch_t<T, TILE32, AK, BKC, 4>(p, count);
    }
    const long long big_tiles = (long long)((p.M + CF::big.BM - 1) / CF::big.BM) * ((p.N + CF::big.BN - 1) / CF::big.BN) * count;
    if (big_tiles * CF::small_div < num_cus) {
        // 64×64 tiles with two k groups of 4 waves (8 waves per workgroup, the groups' sums added through LDS), when
        // they give at least num_cus / 2 tiles: two waves per SIMD hide each other's barrier and load waits without a
        // split-K pass. Measured (TFLOP/s, against the small tiles with split-K): FP32 NN n = 1024 71 → 82, TN 68 → 77,
        // n = 1000 38 → 56, 1024² × K 4096 81 → 98; FP64 n = 1024 44 → 52, n = 1536 38 → 48, 128×4096×128 (the
        // triangular solve's block products) 8.6 → 15.8. FP32 above num_cus tiles loses (n = 1280: 74 → 70), FP64
        // does not. Other FP64 shapes measured at n = 1024 / 1536 against 53.6 / 48.1: four k groups of 2×2 waves
        // 54.0 / 45.1, four of one 64×64 wave 41.9 / 34.9, two of 1×2 waves 48.7, four of 2×1 waves 51.1.
        // A batch (count > 1) cannot split K, so it takes these tiles from num_cus / 4 of them: FP64 128³ × 16 (the
        // triangular solve's 256-row compositions) 12.7 → 8.2 µs on 64 workgroups of 8 waves instead of 32 of 64×128,
        // DTRSM n = 4096 1.458 → 1.443 ms. (The FP64 figures of at most two 32×32 tiles per CU date from before those tiles,
        // which take such products now.)
        if constexpr (sizeof(T) >= 4) {
            const long long t64 = (long long)((p.M + 63) / 64) * ((p.N + 63) / 64) * count;
            const long long need = count > 1 ? (num_cus + 3) / 4 : (num_cus + 1) / 2;
            if (splitk_forced() < 0 && t64 >= need && (sizeof(T) == 8 || t64 <= num_cus))
                return launch_t<T, TILE64, AK, BKC, 2>(p, count);
        }
        return launch_t<T, CF::small, AK, BKC>(p, count);
    }
    // FP64 whose big tiles are exactly half the CUs (K would be split in two, with a reduction pass after): the small
    // tiles instead, when they fill the CUs. MI355X, µs (TFLOP/s): 1024×4096×1024 with beta = 1 (the triangular
    // solve's update of 1024 rows) 152.9 → 141.5 (56.2 → 60.7), 2048³ 268.4 → 258.3 (64.0 → 66.5); DTRSM n = 4096
    // 1.613 → 1.565 ms. 64×64 tiles with two k groups there: 142.8 and 265.9.
    if constexpr (sizeof(T) == 8) {
        const long long ts = (long long)((p.M + CF::small.BM - 1) / CF::small.BM) *
                             ((p.N + CF::small.BN - 1) / CF::small.BN) * count;
        if (splitk_forced() < 0 && count == 1 && big_tiles * 2 == num_cus && ts >= num_cus)
            return launch_t<T, CF::small, AK, BKC>(p, count);
    }
    // FP32 with B k-contiguous has 64×64 big tiles, so a product of exactly num_cus of them lands here: the same
    // two-k-group tiles (NT n = 1024)
    if constexpr (sizeof(T) == 4) {
        const long long t64 = (long long)((p.M + 63) / 64) * ((p.N + 63) / 64) * count;
        if (splitk_forced() < 0 && t64 * 2 >= num_cus && t64 <= num_cus)
            return launch_t<T, TILE64, AK, BKC, 2>(p, count);
    }
    // FP32: 128×128 tiles with two k groups of 2×2 waves (64×64 per wave, 147 KiB of LDS: one workgroup per CU) when
    // their count fills whole rounds of num_cus workgroups (the last round at least 95 % full). Measured (TFLOP/s,
    // against the big tiles above): n = 4096 NN 123 → 125.5, TN 110 → 127.5, NT 123 → 132, n = 2048 NN 118 → 121.5;
    // the odd shape 3000×11008 (2064 tiles, nine rounds with a nearly empty last one) would fall from 117 to 97.
    if constexpr (sizeof(T) == 4) {
        const long long t128 = (long long)((p.M + 127) / 128) * ((p.N + 127) / 128) * count;
        const long long rounds = (t128 + num_cus - 1) / num_cus;
        if (splitk_forced() < 0 && t128 >= num_cus && t128 * 20 >= rounds * num_cus * 19)
            return launch_t<T, TileCfg{128, 128, 2, 2}, AK, BKC, 2>(p, count);
    }
    return launch_t<T, CF::big, AK, BKC>(p, count);
}

}  // namespace g9
#include "hgemm_launch.h"
namespace g9 {

// ---------------- FP32 on direct global→LDS loads ----------------
// Workgroups of KERN (threads each) that one CU holds at once, from the runtime's occupancy query (1 if it fails).
template <auto KERN> static int wgs_per_cu(int threads) {
    static const int occ = [threads] {
        int o = 0;
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(&o, KERN, threads, 0) == hipSuccess && o > 0 ? o : 1;
    }();
    return occ;
}
// k-limited tiles in the paired order: more tiles than CUs, all of them resident at once with two per CU (so that
// workgroups i and i + tiles / 2 run side by side on one CU, each long range beside a short one). With fewer per CU
// the later half starts as CUs free up, and the longest-first order balances better.
static int klim_pair(long long tiles, int per_cu) { return tiles > num_cus && tiles <= 2LL * num_cus && per_cu >= 2; }

}  // namespace g9
#include "sgemm_launch.h"
namespace g9 {

template <class T>
static int launch_typed(const GemmCall &c) {
    using S = typename Mma<T>::Sum;
    GemmParams<S> p;
    p.A = c.A; p.B = c.B; p.C = c.C;
    p.lda = c.lda; p.ldb = c.ldb; p.ldc = c.ldc;
    p.sA = c.sA; p.sB = c.sB; p.sC = c.sC;
    p.M = c.M; p.N = c.N; p.K = c.K;
    p.alpha = (S)c.alpha;
    p.beta = (S)c.beta;
    p.tiles_m = p.tiles_n = 0;
    p.P = nullptr;
    p.kper = 0;
    p.lastk = splitk_forced() >= 0;
    const bool ak = !c.tA, bk = c.tB;   // k-contiguous A: not transposed; k-contiguous B: transposed (stored N×K)
    if (ak) return bk ? launch_layout<T, true, true>(p, c.count) : launch_layout<T, true, false>(p, c.count);
    return bk ? launch_layout<T, false, true>(p, c.count) : launch_layout<T, false, false>(p, c.count);
}

// Triangle of a square product (SYRK, SYR2K): alpha·op(A)·op(B) + beta·C written on the lower (upper) triangle of C
// only. One launch over the T(T+1)/2 square tiles that meet the triangle (T tiles per side), diagonal tiles masked per
// element, each C element rounded once; the two layouts those routines use: A and B both k-contiguous, or both
// mn-contiguous. FP32 and FP64 take 64×64 tiles: at n = 4096 their 2080 tiles keep every CU busy to the end (FP32
// SYRK 0.71 ms, FP64 1.21), where 128×128 tiles (528) left a nearly empty last round (1.02, 1.58).
// FP64 triangles of few tiles and a long K: slices of K, as many as keep four workgroups per CU busy, of at least
// TRI_SLICE_K. A Gram matrix of 1000 features is 136 tiles, half the CUs with one workgroup each.
// MI355X, µs, N×K, unsliced -> sliced: 1000×20000 1474 -> 399, 128×40000 1662 -> 37, 333×7001 421 -> 40, 600×700 52 -> 22,
// 1400×15000 1145 -> 511, 2000×9000 1145 -> 816; the shortest it takes, 64×512, 21.6 -> 15.4.
constexpr int TRI_SLICE_K = 256, TRI_SLICES = 64;
template <class T, int TRI, bool AK, bool BKC, Loads LOADS = UNCHECKED>
static int launch_tri_t(GemmParams<typename Mma<T>::Sum> p) {
    constexpr TileCfg C = sizeof(T) == 2 && LOADS == UNCHECKED ? TileCfg{128, 128, 2, 2} : TILE64;
    if constexpr (LOADS == UNCHECKED) {
        if constexpr (sizeof(T) < 8 && !(AK && BKC))
            if (!unchecked_ok<T>(AK, p.lda) || !unchecked_ok<T>(BKC, p.ldb)) return launch_tri_t<T, TRI, AK, BKC, CHECKED>(p);
        if (!narrow<T, C, AK, BKC>(p)) return launch_tri_t<T, TRI, AK, BKC, WIDE>(p);
    }
    p.tiles_m = p.tiles_n = (p.M + C.BM - 1) / C.BM;
    const long long tiles = (long long)p.tiles_m * (p.tiles_m + 1) / 2;
    if (tiles > 0x7fffffffLL) G9_FAIL(GEN9BLAS_ERR_UNSUPPORTED, "triangle product too large (%d tiles per side)", p.tiles_m);
    if constexpr (sizeof(T) == 8) {
        constexpr int BK = 128 / (int)sizeof(T);
        int ns = (int)std::min<long long>({4LL * num_cus / tiles, p.K / TRI_SLICE_K, TRI_SLICES});
        void *P = nullptr;
        if (ns > 1 && splitk_forced() < 0) {   // fewer slices, or none, where the work space could not be had
            size_t work;
            P = splitk_workspace(&work);
            ns = (int)std::min<size_t>(ns, work / ((size_t)p.M * p.M * sizeof(T)));
        }
        if (ns > 1 && P) {
            auto q = p;
            q.kper = ((p.K + ns - 1) / ns + BK - 1) / BK * BK;
            ns = (p.K + q.kper - 1) / q.kper;
            q.C = P;
            q.ldc = p.M;
            q.sA = q.kper * (AK ? 1 : p.lda);
            q.sB = q.kper * (BKC ? 1 : p.ldb);
            q.sC = (long long)p.M * p.M;
            q.alpha = 1;
            q.beta = 0;
            hipLaunchKernelGGL((gemm_kernel<T, C.BM, C.BN, C.WM, C.WN, AK, BKC, false, TRI, 0, 1, LOADS>),
                               dim3((unsigned)tiles, (unsigned)ns), dim3(C.WM * C.WN * 64), 0, stream, q);
            G9_HIP(hipGetLastError());
            hipLaunchKernelGGL((tri_split_sum<T, T>), dim3((unsigned)((p.M + 255) / 256), (unsigned)p.M), dim3(256), 0, stream,
                               (const T *)P, (T *)p.C, p.ldc, p.M, ns, TRI == 1, p.alpha, p.beta);
            G9_HIP(hipGetLastError());
            return 0;
        }
    }
    hipLaunchKernelGGL((gemm_kernel<T, C.BM, C.BN, C.WM, C.WN, AK, BKC, false, TRI, 0, 1, LOADS>), dim3((unsigned)tiles),
                       dim3(C.WM * C.WN * 64), 0, stream, p);
    G9_HIP(hipGetLastError());
    return 0;
}
template <class T, bool AK, bool BKC>
static int launch_tri_layout(const GemmParams<typename Mma<T>::Sum> &p, bool lower) {
    return lower ? launch_tri_t<T, 1, AK, BKC>(p) : launch_tri_t<T, 2, AK, BKC>(p);
}
template <class T>
static int launch_tri_typed(const GemmCall &c, bool lower) {
    using S = typename Mma<T>::Sum;
    GemmParams<S> p;
    p.A = c.A; p.B = c.B; p.C = c.C;
    p.lda = c.lda; p.ldb = c.ldb; p.ldc = c.ldc;
    const bool batch = c.count > 1;
    p.sA = batch ? c.sA : 0; p.sB = batch ? c.sB : 0; p.sC = batch ? c.sC : 0;
    p.M = c.M; p.N = c.N; p.K = c.K;
    p.alpha = (S)c.alpha;
    p.beta = (S)c.beta;
    p.tiles_m = p.tiles_n = 0;
    p.P = nullptr;
    p.kper = 0;
    p.lastk = splitk_forced() >= 0;
    if (!c.tA && c.tB) return launch_tri_layout<T, true, true>(p, lower);
    if (c.tA && !c.tB) return launch_tri_layout<T, false, false>(p, lower);
    G9_FAIL(GEN9BLAS_ERR_UNSUPPORTED, "triangle product: layout tA=%d tB=%d", c.tA, c.tB);
}
int launch_gemm_tri(const GemmCall &c, bool lower) {
    if (c.M != c.N || c.count != 1) G9_FAIL(GEN9BLAS_ERR_UNSUPPORTED, "triangle product: %d×%d, batch %d", c.M, c.N, c.count);
    switch (c.type) {
    case GEN9BLAS_H:
    case GEN9BLAS_HS: return launch_tri_typed<f16>(c, lower);
    case GEN9BLAS_S: {
        int rc = 0;
        return sg_tri(c, lower, &rc) ? rc : launch_tri_typed<float>(c, lower);
    }
    case GEN9BLAS_D: return launch_tri_typed<double>(c, lower);
    }
    G9_FAIL(GEN9BLAS_ERR_UNSUPPORTED, "type %d unavailable", c.type);
}

// Product with a triangular operand (TRMM on the explicit triangular matrix, TRSM's leaf products): each tile's k
// range is cut to where the triangle is non-zero (klim as gemm_kernel's KLIM), one launch over every tile of C,
// longest ranges dispatched first; the small tiles when the big ones are fewer than the CUs. Layout NN only (both
// operands as stored), one product.
template <class T, TileCfg C, int KLIM, int KG = 1, Loads LOADS = UNCHECKED>
static int launch_klim_t(GemmParams<typename Mma<T>::Sum> p, int count) {
    if constexpr (LOADS == UNCHECKED)
        if (!narrow<T, C, true, false>(p)) return launch_klim_t<T, TILE64, KLIM, 1, WIDE>(p, count);
    p.tiles_m = (p.M + C.BM - 1) / C.BM;
    p.tiles_n = (p.N + C.BN - 1) / C.BN;
    const long long tiles = (long long)p.tiles_m * p.tiles_n;
    if (tiles > 0x7fffffffLL) G9_FAIL(GEN9BLAS_ERR_UNSUPPORTED, "gemm grid too large (%d × %d tiles)", p.tiles_m, p.tiles_n);
    constexpr auto kern = gemm_kernel<T, C.BM, C.BN, C.WM, C.WN, true, false, false, 0, KLIM, KG, LOADS>;
    p.kpair = count == 1 && klim_pair(tiles, wgs_per_cu<kern>(C.WM * C.WN * 64 * KG));
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles, (unsigned)count), dim3(C.WM * C.WN * 64 * KG), 0, stream, p);
    G9_HIP(hipGetLastError());
    return 0;
}
template <class T>
static int launch_klim_typed(const GemmCall &c, int klim) {
    using S = typename Mma<T>::Sum;
    GemmParams<S> p;
    p.A = c.A; p.B = c.B; p.C = c.C;
    p.lda = c.lda; p.ldb = c.ldb; p.ldc = c.ldc;
    const bool batch = c.count > 1;
    p.sA = batch ? c.sA : 0; p.sB = batch ? c.sB : 0; p.sC = batch ? c.sC : 0;
    p.M = c.M; p.N = c.N; p.K = c.K;
    p.alpha = (S)c.alpha;
    p.beta = (S)c.beta;
    p.tiles_m = p.tiles_n = 0;
    p.P = nullptr;
    p.kper = 0;
    p.lastk = splitk_forced() >= 0;
    // tile class: FP16 the big tiles when they are at least the CUs; FP32 / FP64 the first of big, small and (FP64)
    // 64×64 that makes two workgroups per CU or more, so that long and short k ranges can share the CUs
    using CF = Cfg<T, true, false>;
    const auto ntiles = [&](TileCfg t) {
        return (long long)((c.M + t.BM - 1) / t.BM) * ((c.N + t.BN - 1) / t.BN) * c.count;
    };
    constexpr bool half = sizeof(T) == 2, dbl = sizeof(T) == 8;
    const long long want = half ? num_cus : 2LL * num_cus;
    // FP64 below that: 32×32 tiles with four k groups up to two workgroups per CU, then 32×64 with two. MI355X, µs,
    // 64×64 -> these: 1024×500 43.9 -> 20.0, 512×500 22.0 -> 11.2, 1024×16 39.4 -> 15.6; 1024×1000 44.2 -> 26.9 (32×32:
    // 32.3); 1024×2048 45.4 against 48.0, 512×4096 27.6 against 29.3.
    constexpr TileCfg half_wide{32, 64, 1, 2};
    // A forced split-K asks for one summation order: 64×64 tiles (FP32's small ones) without k groups, as the k range of
    // a row, and so its order of k-steps, follows the tile.
    const bool fixed = !half && splitk_forced() >= 0;
    const int cls = fixed ? (dbl ? 2 : 1) : ntiles(CF::big) >= want ? 0 : (!dbl || ntiles(CF::small) >= want) ? 1 : 2;
    const auto go = [&](auto kc) -> int {
        constexpr int K = decltype(kc)::value;
        if constexpr (!dbl)
            if (!unchecked_ok<T>(false, p.ldb)) return launch_klim_t<T, TILE64, K, 1, CHECKED>(p, c.count);
        if (cls == 0) return launch_klim_t<T, CF::big, K>(p, c.count);
        if constexpr (dbl) {
            if (!fixed && ntiles(TILE32) <= 2LL * num_cus) return launch_klim_t<T, TILE32, K, 4>(p, c.count);
            if (!fixed && ntiles(half_wide) <= 2LL * num_cus) return launch_klim_t<T, half_wide, K, 2>(p, c.count);
            if (cls == 2) return launch_klim_t<T, TILE64, K>(p, c.count);
        }
        return launch_klim_t<T, CF::small, K>(p, c.count);
    };
    switch (klim) {
    case 1: return go(std::integral_constant<int, 1>());
    case 2: return go(std::integral_constant<int, 2>());
    case 3: return go(std::integral_constant<int, 3>());
    case 4: return go(std::integral_constant<int, 4>());
    }
    G9_FAIL(GEN9BLAS_ERR_UNSUPPORTED, "k-limited product: mode %d", klim);
}
int launch_gemm_klim(const GemmCall &c, int klim) {
    if (c.tA || c.tB || c.count < 1) G9_FAIL(GEN9BLAS_ERR_UNSUPPORTED, "k-limited product: layout tA=%d tB=%d, batch %d", c.tA, c.tB, c.count);
    switch (c.type) {
    case GEN9BLAS_H:
    case GEN9BLAS_HS: return launch_klim_typed<f16>(c, klim);
    case GEN9BLAS_S: {
        int rc = 0;
        return sg_klim(c, klim, &rc) ? rc : launch_klim_typed<float>(c, klim);
    }
    case GEN9BLAS_D: return launch_klim_typed<double>(c, klim);
    }
    G9_FAIL(GEN9BLAS_ERR_UNSUPPORTED, "type %d unavailable", c.type);
}

int launch_gemm(const GemmCall &c) {
    switch (c.type) {
    case GEN9BLAS_H:
    case GEN9BLAS_HS: {
        int rc = 0;
        return launch_hgemm_tiles(c, &rc) ? rc : launch_typed<f16>(c);
    }
    case GEN9BLAS_S: {
        int rc = 0;
        return launch_sgemm_direct(c, &rc) ? rc : launch_typed<float>(c);
    }
    case GEN9BLAS_D: return launch_typed<double>(c);
    }
    G9_FAIL(GEN9BLAS_ERR_UNSUPPORTED, "type %d unavailable", c.type);
}

}  // namespace g9
