// Host side of the FP32 GEMM on direct global→LDS loads (sgemm_kernel.h): which products it takes, their tiles and their
// split of K, the triangle and k-limited modes of the level-3 routines. Part of gemm_kernels.hip.
// Against the general kernel that served ragged products before, with checked loads in every k-step and whole-tile interiors
// (µs): 1000³ 37.4 → 25.0, 64 × 250³ 46.1 → 27.7, 141×3840×3712 TN 205 → 60, 6192×192×5910 NT 413 → 143, 1512×362×738
// 43.4 → 19.5.
//
// Tile configurations, with rates on MI355X (TFLOP/s, sustained): 128×256, 8 waves of 64×64, two stages, sums blocked per
// 128 k: n = 4096 NN 144.9, NT 144.3, 8192×8192×2048 144.1 (three stages 142.6; blocks of 32 k 134.3, 64 k 140.3, 256 k
// 142.6; 256×128 tiles 142.7). 128×128, 8 waves of 64×32, three stages: n = 2048 133-134 (4 waves of 64×64 129.7).
// 64×64, 4 waves of 32×32, four stages, sums blocked per 256 k: n = 2048 137, n = 1024 102.6 (three stages 94.0, six 93.0,
// eight 92.2; 128-k blocks 101.9, 32-k 90.9). 64×128 and 128×64, 4 waves of 32×64 (64×32), three stages:
// 2386×1512×1920 120.5 µs against 121.1 on 64×64 and 122.1 on 128×128 tiles, 3000×3000×150 42.6 against 43.1 and 46.5.
#pragma once
#include "sgemm_kernel.h"
#include <stdlib.h>
#include <string.h>
#include <algorithm>
#include <cmath>

namespace g9 {
namespace sgl {

constexpr int KB = 32;   // k per k-step
// ns: time per k of a 64×64 share of the tile, for cost(); per_cu: workgroups that share a CU
struct SgCfg { int BM, BN, WM, WN, NS, BLK; double ns; int per_cu; };
constexpr SgCfg CFG[] = {{128, 256, 2, 4, 2, 4, 14.4, 1}, {128, 128, 2, 4, 3, 4, 14.8, 1}, {64, 64, 2, 2, 4, 8, 14.8, 2},
                         {64, 128, 2, 2, 3, 4, 14.8, 2}, {128, 64, 2, 2, 3, 4, 14.8, 2}};
constexpr int NCFG = sizeof CFG / sizeof CFG[0];
struct Choice { int cfg, slices; double us; };

static int slices_of(int K, int s, int &kper) {
    kper = std::max(((K + s - 1) / s + KB - 1) / KB * KB, 2 * KB);
    return (K + kper - 1) / kper;
}
// Estimated time (µs) of `tiles` tiles of a configuration in ns slices of kper k: the launch, the most loaded CU's tiles at
// the matrix cores' rate, a fixed part for each round of tiles that share a CU, and for slices the second kernel and
// their sums written and read. Constants fitted to 29 products (K 100 to 20000, 100 to 8000 rows, batches, whole and
// ragged, every layout), timed with every configuration and 1-24 slices: the choice is the fastest or within 2 % of it for
// 27 of them, within 7 % for all. A few (µs, chosen / others): 500³ 64×64 in 3 slices 10.2 / unsplit 12.1; 130×130×5000
// 64×64 in 16-24 slices 16.9 / in 4 24; 64 × 256³ 128×128 24.8 / 64×64 27.4; 245 × 144×64×264 64×64 25.5 / 128×128 48.5.
static double cost(const SgCfg &g, long long tiles, int kper, int ns) {
    const double per_cu = (double)(tiles * ns) / num_cus, area = (double)g.BM * g.BN / 4096;
    double t = 5.4 + std::max(1.0, std::ceil(per_cu)) * area * g.ns * 1e-3 * kper + 3.4 * std::ceil(per_cu / g.per_cu);
    if (ns > 1) t += 0.8 + (double)(ns * tiles) * g.BM * g.BN * 8 / 1e7;
    return t;
}
// The cheapest configuration and split of K into slices that fit `work` bytes; tri: the tiles of a triangle of side M
// (square tiles only); big: 128×256 tiles may be taken (their edge-capable variant would need more registers than a wave
// has).
static Choice choose(const GemmCall &c, size_t work, bool tri, bool big) {
    static constexpr int SLICES[] = {1, 2, 3, 4, 6, 8, 12, 16, 24};
    Choice best{2, 1, 1e30};
    for (int i = 0; i < NCFG; i++) {
        const SgCfg &g = CFG[i];
        // a triangle that no whole tiles fill: 128×128 tiles lose half of each on the diagonal, and on this kernel they
        // were slower throughout (2000×200 22.1 µs against 20.0, 5000×160 50.8 against 40.3)
        if ((tri && (g.BM != g.BN || (g.BM == 128 && c.M % 64))) || (i == 0 && !big)) continue;
        const long long tm = (c.M + g.BM - 1) / g.BM, tn = (c.N + g.BN - 1) / g.BN;
        const long long tiles = (tri ? tm * (tm + 1) / 2 : tm * tn) * c.count;
        for (const int s : SLICES) {
            int kper;
            const int ns = s == 1 ? 1 : slices_of(c.K, s, kper);
            if (s == 1) kper = (c.K + KB - 1) / KB * KB;
            if (s > 1 && (i == 0 || kper < 4 * KB || tiles * s > 5LL * num_cus ||
                          (size_t)(ns * tiles) * g.BM * g.BN * sizeof(float) > work)) break;
            const double t = cost(g, tiles, kper, ns);
            if (t < best.us) best = Choice{i, ns, t};
        }
    }
    return best;
}

// TRI: 0 plain, 1 lower, 2 upper triangle (square tiles). EDGE as in the kernel; slices > 1 needs p.P.
template <int I, bool AK, bool BKC, int TRI, bool EDGE>
static int launch_cfg(sg::Params p, int count, int slices) {
    constexpr SgCfg G = CFG[I];
    p.tiles_m = (p.M + G.BM - 1) / G.BM;
    p.tiles_n = (p.N + G.BN - 1) / G.BN;
    const unsigned tiles = TRI ? (unsigned)((long long)p.tiles_m * (p.tiles_m + 1) / 2) : (unsigned)(p.tiles_m * p.tiles_n);
    const dim3 block(G.WM * G.WN * 64);
    if constexpr (EDGE) {
        if (slices > 1 && p.P) {
            const int ns = slices_of(p.K, slices, p.kper);
            hipLaunchKernelGGL((sg::sgemm_kernel<G.BM, G.BN, G.WM, G.WN, G.NS, AK, BKC, G.BLK, TRI, 0, false, true, true>),
                               dim3(tiles, (unsigned)ns), block, 0, stream, p);
            G9_HIP(hipGetLastError());
            constexpr int PER = G.BM * G.BN / 256;   // 256 elements of C per wave
            hipLaunchKernelGGL((sg::split_sum<G.BM, G.BN, G.WM, G.WN, TRI>), dim3((unsigned)(((long long)tiles * PER + 3) / 4)),
                               dim3(256), 0, stream, p, ns, (int)tiles);
            G9_HIP(hipGetLastError());
            return 0;
        }
    }
    hipLaunchKernelGGL((sg::sgemm_kernel<G.BM, G.BN, G.WM, G.WN, G.NS, AK, BKC, G.BLK, TRI, 0, false, EDGE>),
                       dim3(tiles, (unsigned)count), block, 0, stream, p);
    G9_HIP(hipGetLastError());
    return 0;
}
template <bool AK, bool BKC>
static int launch_plain(const sg::Params &p, int count, Choice ch, bool whole) {
    if (whole && ch.slices == 1) {
        switch (ch.cfg) {
        case 0: return launch_cfg<0, AK, BKC, 0, false>(p, count, 1);
        case 1: return launch_cfg<1, AK, BKC, 0, false>(p, count, 1);
        case 2: return launch_cfg<2, AK, BKC, 0, false>(p, count, 1);
        }
    }
    switch (ch.cfg) {
    case 1: return launch_cfg<1, AK, BKC, 0, true>(p, count, ch.slices);
    case 3: return launch_cfg<3, AK, BKC, 0, true>(p, count, ch.slices);
    case 4: return launch_cfg<4, AK, BKC, 0, true>(p, count, ch.slices);
    }
    return launch_cfg<2, AK, BKC, 0, true>(p, count, ch.slices);
}
template <int TRI, bool AK, bool BKC>
static int launch_tri(const sg::Params &p, Choice ch, bool whole) {
    if (whole && ch.slices == 1)
        return ch.cfg == 1 ? launch_cfg<1, AK, BKC, TRI, false>(p, 1, 1) : launch_cfg<2, AK, BKC, TRI, false>(p, 1, 1);
    return ch.cfg == 1 ? launch_cfg<1, AK, BKC, TRI, true>(p, 1, ch.slices) : launch_cfg<2, AK, BKC, TRI, true>(p, 1, ch.slices);
}

}  // namespace sgl

static sg::Params sg_params(const GemmCall &c) {
    sg::Params p;
    p.A = reinterpret_cast<const float *>(c.A);
    p.B = reinterpret_cast<const float *>(c.B);
    p.C = reinterpret_cast<float *>(c.C);
    p.lda = c.lda; p.ldb = c.ldb; p.ldc = c.ldc;
    p.sA = c.sA; p.sB = c.sB; p.sC = c.sC;
    p.M = c.M; p.N = c.N; p.K = c.K;
    p.tiles_m = p.tiles_n = 0;
    p.alpha = (float)c.alpha;
    p.beta = (float)c.beta;
    return p;
}
// The kernel takes operands at element alignment, lane offsets inside a tile being 32-bit (lane_span), and more than one
// k-step of k (exactly one when no operand row ends inside a 16-byte chunk): the k-step it takes through registers needs a
// direct one beside it. GEN9BLAS_SGEMM=generic and a forced split-K (GEN9BLAS_SPLITK) ask for the general kernel.
static bool sgemm_direct_ok(const GemmCall &c) {
    static const bool generic = [] {
        const char *e = getenv("GEN9BLAS_SGEMM");
        return e && !strcmp(e, "generic");
    }();
    if (generic || splitk_forced() >= 0 || c.count > 65535 || std::min(c.lda, c.ldb) < 4) return false;
    if (lane_span(!c.tA, c.lda * 4, c.M, sgl::KB) >= (1LL << 32) || lane_span(c.tB, c.ldb * 4, c.N, sgl::KB) >= (1LL << 32)) return false;
    return c.K > sgl::KB || (c.K == sgl::KB && !(c.tA && c.M % 4) && !(!c.tB && c.N % 4));
}
// 16-byte aligned operands and row strides, K whole k-steps: what the whole-tile variants take, which check and mask
// nothing.
static bool sgemm_tiles_ok(const GemmCall &c) {
    if (!sgemm_direct_ok(c) || c.K % sgl::KB) return false;
    const auto al16 = [&](const void *x, long long ld, long long s) {
        return (uintptr_t)x % 16 == 0 && ld % 4 == 0 && (c.count == 1 || s % 4 == 0);
    };
    return al16(c.A, c.lda, c.sA) && al16(c.B, c.ldb, c.sB) && al16(c.C, c.ldc, c.sC);
}
// The whole-tile variants sum blocks of 128 k (64×64 tiles: 256 k), which is a little faster than the edge-capable tiles'
// blocks of 32 and rounds a little more (1000³: 2.9e-7 against 1.3e-7 of the result), so they serve the products that fill
// the chip with them and no others: the longest block of the first class whose whole tiles fill the CUs (128×128: twice)
// and cover 90 % of C, 0 when there is none.
static int whole_block(const GemmCall &c) {
    for (int i = 0; i < 3; i++) {
        const sgl::SgCfg &g = sgl::CFG[i];
        const long long tm = c.M / g.BM, tn = c.N / g.BN;
        if (tm * tn * c.count >= (i == 1 ? 2LL : 1LL) * num_cus && (double)(tm * g.BM) * (tn * g.BN) >= 0.9 * (double)c.M * c.N)
            return g.BLK;
    }
    return 0;
}
// Parameters, with the work space of split products.
static sg::Params sg_work(const GemmCall &c, bool batch, size_t &work) {
    sg::Params p = sg_params(c);
    work = 0;
    if (batch) return p;
    p.sA = p.sB = p.sC = 0;
    p.P = reinterpret_cast<float *>(splitk_workspace(&work));
    return p;
}

// Triangle of an FP32 square product (NT or TN). K is split where the triangle leaves CUs idle: XᵀX of 20000×1000 takes
// 220 µs (1137 on 136 unsplit tiles of 64×64), of 13321×896 95 (466).
// A rank-K update with a short K of a triangle that fills the chip is bound by C, which the general kernel's four workgroups
// per CU write faster: 2000×64 8.0 against 11.7, 5000×128 38 against 51, at β = 0.5 46 against 62 (1500×128 9.9 either way).
static bool sg_tri(const GemmCall &c, bool lower, int *rc) {
    if (c.M != c.N || c.count != 1 || !sgemm_direct_ok(c) || c.tA == c.tB) return false;
    const long long side = (c.M + 63) / 64;
    if (c.K <= 128 && side * (side + 1) / 2 > 2LL * num_cus) return false;
    size_t work;
    const sg::Params p = sg_work(c, false, work);
    const sgl::Choice ch = sgl::choose(c, work, true, false);
    // whole tiles (sums blocked per 128 or 256 k, as whole_block) where they fill the CUs, 64×64 ones unless 128×128 fill
    // their last round as well
    const long long s64 = c.M / 64, s128 = c.M / 128, t64 = s64 * (s64 + 1) / 2, t128 = s128 * (s128 + 1) / 2;
    const auto fill = [](long long t) { return (double)t / (double)(((t + num_cus - 1) / num_cus) * num_cus); };
    const bool big = c.M % 128 == 0 && t128 >= num_cus && (c.M % 64 || t64 < num_cus || fill(t128) >= fill(t64));
    const bool whole = sgemm_tiles_ok(c) && c.M % sgl::CFG[ch.cfg].BM == 0 && (ch.cfg == 1 ? big || t64 >= num_cus : !big && t64 >= num_cus);
    if (c.tB) *rc = lower ? sgl::launch_tri<1, true, true>(p, ch, whole) : sgl::launch_tri<2, true, true>(p, ch, whole);
    else *rc = lower ? sgl::launch_tri<1, false, false>(p, ch, whole) : sgl::launch_tri<2, false, false>(p, ch, whole);
    return true;
}

// k-limited mode (KLIM): one product, whole tiles (the callers check), `tiles` workgroups.
template <int BM, int BN, int WM, int WN, int NS, int BLK, bool AK, bool BKC, int TRI, int KLIM>
static int launch_sg_mode(const sg::Params &p0, long long tiles, int count = 1) {
    constexpr auto kern = sg::sgemm_kernel<BM, BN, WM, WN, NS, AK, BKC, BLK, TRI, KLIM>;
    sg::Params p = p0;
    p.tiles_m = p.M / BM;
    p.tiles_n = p.N / BN;
    if constexpr (KLIM != 0) p.kpair = count == 1 && klim_pair(tiles, wgs_per_cu<kern>(WM * WN * 64));
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles, (unsigned)count), dim3(WM * WN * 64), 0, stream, p);
    G9_HIP(hipGetLastError());
    return 0;
}
// k-limited FP32 NN product (or strided batch of them) on the whole-tile kernel (TRMM, the triangular solves): the
// plain products' classes, whole tiles only. A batch takes the big classes only with two tiles per CU or more, so
// that tiles of long and short k ranges share the CUs (TRSV's E_q = inv(D_q)·C_q, 512³ × 31: 128×128 tiles 80 µs
// in a kernel trace; on 64×64 tiles the n = 16384 solve takes 385 against 400 µs).
template <int KLIM>
static bool sg_klim_mode(const GemmCall &c, int *rc) {
    const sg::Params p = sg_params(c);
    const long long t0 = (long long)(c.M / 128) * (c.N / 256), t1 = (long long)(c.M / 128) * (c.N / 128),
                    t2 = (long long)(c.M / 64) * (c.N / 64), nb = c.count;
    const long long want = nb > 1 ? 2LL * num_cus : num_cus;
    if (c.M % 128 == 0 && c.N % 256 == 0 && t0 * nb >= want)
        *rc = launch_sg_mode<128, 256, 2, 4, 2, 4, true, false, 0, KLIM>(p, t0, c.count);
    else if (c.M % 128 == 0 && c.N % 128 == 0 && t1 * nb >= want)
        *rc = launch_sg_mode<128, 128, 2, 4, 3, 4, true, false, 0, KLIM>(p, t1, c.count);
    else if (c.M % 64 == 0 && c.N % 64 == 0 && t2 * nb >= num_cus)
        *rc = launch_sg_mode<64, 64, 2, 2, 4, 8, true, false, 0, KLIM>(p, t2, c.count);
    else return false;
    return true;
}
static bool sg_klim(const GemmCall &c, int klim, int *rc) {
    // the k range of every tile is non-empty only when K spans the triangular operand's order
    if (c.count < 1 || c.tA || c.tB || !sgemm_tiles_ok(c) || (klim <= 2 ? c.K != c.M : c.K != c.N)) return false;
    switch (klim) {
    case 1: return sg_klim_mode<1>(c, rc);
    case 2: return sg_klim_mode<2>(c, rc);
    case 3: return sg_klim_mode<3>(c, rc);
    case 4: return sg_klim_mode<4>(c, rc);
    }
    return false;
}


// A large product whose rows do not fill whole 128×256 tiles (two rounds of them or more, whole columns): the whole tiles,
// then the bottom strip of r rows on 64×64 tiles shifted up onto the last ⌈r/64⌉·64 rows, storing only its own r. Larger
// tiles are worth it there: 3000×11008×4096 NT β = 0.5 takes 1.97 ms, in one launch 2.01 on 64×64 tiles and 2.41 on
// 128×256. Returns false, with nothing launched, when it does not apply or `us`, another way's estimate, is lower.
static bool sg_strip(const GemmCall &c, const sg::Params &p0, double us, int *rc) {
    constexpr sgl::SgCfg big = sgl::CFG[0], small = sgl::CFG[2];
    const int Mi = c.M / big.BM * big.BM, r = c.M - Mi, Ms = (r + 63) / 64 * 64;
    if (c.count != 1 || r == 0 || Ms > c.M || c.N % big.BN || (c.tA && (c.M - Ms) % 4) || !sgemm_tiles_ok(c)) return false;
    const long long tiles = (long long)(Mi / big.BM) * (c.N / big.BN), strip = (long long)(Ms / 64) * (c.N / 64);
    if (tiles < 2LL * num_cus || sgl::cost(big, tiles, c.K, 1) + sgl::cost(small, strip, c.K, 1) - 5.4 >= us) return false;
    sg::Params p = p0, s = p0;
    p.M = Mi;
    s.A += c.tA ? (long long)(c.M - Ms) : (long long)(c.M - Ms) * c.lda;
    s.C += (long long)(c.M - Ms) * c.ldc;
    s.M = Ms;
    s.m_skip = Ms - r;
    s.tiles_m = Ms / 64;
    s.tiles_n = c.N / 64;
    const auto go = [&](auto ak, auto bk) -> int {
        constexpr bool AK = decltype(ak)::value, BKC = decltype(bk)::value;
        G9_TRY((sgl::launch_cfg<0, AK, BKC, 0, false>(p, 1, 1)));
        hipLaunchKernelGGL((sg::sgemm_kernel<64, 64, 2, 2, 4, AK, BKC, 8, 0, 0, true>), dim3((unsigned)strip), dim3(256), 0,
                           stream, s);
        G9_HIP(hipGetLastError());
        return 0;
    };
    using Y = std::true_type;
    using N = std::false_type;
    if (c.tA) *rc = c.tB ? go(N(), Y()) : go(N(), N());
    else *rc = c.tB ? go(Y(), Y()) : go(Y(), N());
    return true;
}

// FP32 products on this kernel. False, with nothing launched, for those it does not take.
// Not NT with a short K whose rows of C are not whole 64-byte sectors: C bounds it, and the general kernel writes it
// faster (β = 0.5, K = 33: 1500² 9.7 against 12.9, 3000² 23 against 32, 5000² 52 against 72, 1000² 5 % less; with whole
// sectors, 2000² or 4096², 12 % more). From K = 128 on its one running sum would round more than the two here.
static bool launch_sgemm_direct(const GemmCall &c, int *rc) {
    if (!sgemm_direct_ok(c) || (!c.tA && c.tB && c.K < 128 && c.ldc % 16)) return false;
    const bool batch = c.count > 1;
    size_t work;
    const sg::Params p = sg_work(c, batch, work);
    const bool tiles_ok = sgemm_tiles_ok(c);
    const int block = tiles_ok ? whole_block(c) : 0;
    const sgl::Choice ch = sgl::choose(c, work, false, block >= sgl::CFG[0].BLK && c.M % 128 == 0 && c.N % 256 == 0);
    const sgl::SgCfg &g = sgl::CFG[ch.cfg];
    if ((long long)((c.M + g.BM - 1) / g.BM) * ((c.N + g.BN - 1) / g.BN) > 0x7fffffffLL) return false;
    if (sg_strip(c, p, ch.us, rc)) return true;
    const bool whole = tiles_ok && c.M % g.BM == 0 && c.N % g.BN == 0 && g.BLK <= block;
    if (c.tA) *rc = c.tB ? sgl::launch_plain<false, true>(p, c.count, ch, whole) : sgl::launch_plain<false, false>(p, c.count, ch, whole);
    else *rc = c.tB ? sgl::launch_plain<true, true>(p, c.count, ch, whole) : sgl::launch_plain<true, false>(p, c.count, ch, whole);
    return true;
}

}  // namespace g9
