// Host side of the FP16 GEMM on direct global→LDS loads (hgemm_kernel.h): which products it takes, their tiles and their
// split of K. Part of gemm_kernels.hip: one code object for the GEMM kernels, loaded as a whole with the first of them.
//
// Tile configurations come from sweeps on MI355X with N(0,1) FP16 inputs, timed after 1.5 s of the same load (the clock
// settles under the board's power limit; shorter runs see its ramp), every variant bit-exact on small integers:
// - 256×256 tiles, 8 waves of 128×64 (2×4), two stages of 64 k. n = 4096 NN 1314-1324 TFLOP/s (8 waves of 64×128:
//   1276-1286; 4 waves of 128×128: 1243-1246, at 2.03 GHz against 1.79-1.81; the same 8 waves on 32x32x16 MFMAs:
//   1166-1176); TN 1249, NT 1339, TT 1267 (32x32x16: 1180-1188);
// - 128×128, 8 waves of 64×32 (2×4), three stages. n = 2048 NN 835 (4 waves of 64×64 with 3 or 4 stages: 798-807;
//   32x32x16 tiles: 795), NT 845 (767), TN and TT 800-804 (800-802);
// - 64×64, 4 waves of 32×32, three stages, fragments read one k-step ahead: n = 1024 NT 399.9 (four stages 390.6, two
//   303.6, no read-ahead 378.1), NN 400.7 (its 64-wide mn-contiguous B rows swizzled by mnswz). Before them 32×128
//   tiles, NN 382.8; 128×128 tiles for a transposed A, TN 212.6 → 365.5, TT 215.3 → 393.1. Time per call against K at
//   M = N = 1024 is about 2-3 µs plus 0.26 µs per k-step of 64: the k-step's latency chain sets the rate;
// - 256×192 (192×256), 8 waves of 64×96 (96×64), two stages, and 256×128 (128×256), 8 waves of 64×64, three stages, for
//   tile counts that leave the larger tiles' last round, or the only one, part empty (µs): 1000×11008×4096 NT 94.5 on
//   232 tiles of 256×192 against 100.7 on 172 of 256×256, 114 on 688 of 128×128 and 109 on 344 of 256×128; 2504³ NT 60.4
//   on 200 of 128×256 against 66.2 on 400 of 128×128. A 192-wide operand must be k-contiguous.
#pragma once
#include "hgemm_kernel.h"
#include <stdlib.h>
#include <string.h>
#include <algorithm>
#include <cmath>

namespace g9 {

// Bytes that the direct copies' lane offsets reach over inside a tile of at most 256 rows: the rows of a k-contiguous
// operand of MN rows, the k rows of a k-step otherwise (ldb: row stride in bytes). They are 32-bit.
static long long lane_span(bool kc, long long ldb, int MN, int kb) { return (kc ? std::min(256, MN) : kb) * ldb; }

namespace hgl {

constexpr int KB = 64;   // k per k-step
// For choose(): ns, time per k of a round of one tile per CU on the whole chip; fix, the rest of a round (µs); st, µs per MB
// of C stored
struct HgCfg { int BM, BN, WM, WN, NS; bool RA; double ns, fix, st; };
constexpr HgCfg CFG[] = {{256, 256, 2, 4, 2, false, 25, 3.1, 0.062}, {128, 128, 2, 4, 3, false, 8.1, 1.8, 0.037},
                         {64, 64, 2, 2, 3, true, 3.3, 1.8, 0}, {256, 192, 4, 2, 2, false, 22, 2.1, 0.064},
                         {192, 256, 2, 4, 2, false, 22, 2.1, 0.064}, {256, 128, 4, 2, 3, false, 13.07, 3, 0.044},
                         {128, 256, 2, 4, 3, false, 13, 3, 0.044}};
constexpr int NCFG = sizeof CFG / sizeof CFG[0];

static long long tiles_of(const HgCfg &g, int M, int N) { return (long long)((M + g.BM - 1) / g.BM) * ((N + g.BN - 1) / g.BN); }

struct Choice { int cfg, slices; };
// The configuration and number of K slices with the smallest estimated time (µs): a launch; rounds of one tile per CU
// (64×64: two share a CU, one alone takes two thirds of their time), each a fixed part and the tile's time per k, less where
// part of the chip idles (the board's power limit leaves the rest a higher clock); C written by the larger tiles, which
// costs most where its rows are not whole 128-byte lines; for slices, the second kernel, its pass over each slice, and the
// FP32 sums written and read.
// The constants are a fit to the order of 392 products (K 64 to 11008, 17 to 20000 rows, batches, whole and ragged, NN /
// NT / TN), each timed with every configuration and 1-16 slices on operands in the last-level cache and rotated beyond it:
// by the geometric mean of both the choice is 0.6 % from the fastest on average, and within 22 % for all. A few (µs,
// in the cache and beyond it, chosen / others): 48×4096×4096 NT 64×64 in 4 slices 10.7 and 12.7 / unsplit 21 and 23;
// 600×4096×11008 128×256 in 3 slices 74 / 128×128 unsplit 103; 256×1024×1024 64×64 5.4 and 8.2 / in 3 slices 7.5 and 8.5;
// 1280³ 64×64 9.1 and 11.7 / 128×128 11.3 and 14.4; 5000×5000×64 64×64 or 128×128 27 and 31 / 256×256 41 and 48. Slices hold
// at least 256 k and fit the `work` bytes of the split-K work space.
static Choice choose(const GemmCall &c, size_t work) {
    static constexpr int SLICES[] = {1, 2, 3, 4, 6, 8, 12, 16};
    const double mn = (double)c.M * c.N, c_mb = 2e-6 * c.count * mn * (c.ldc % 64 ? 7 : 1);
    Choice best{0, 1};
    double t_best = 1e30;
    for (int i = 0; i < NCFG; i++) {
        const HgCfg &g = CFG[i];
        if ((g.BN == 192 && !c.tB) || (g.BM == 192 && c.tA)) continue;
        const long long tiles = tiles_of(g, c.M, c.N) * c.count;
        for (const int s : SLICES) {
            const int kper = ((c.K + s - 1) / s + KB - 1) / KB * KB, ns = (c.K + kper - 1) / kper;
            if (s > 1 && (kper < 256 || tiles * s > 3LL * num_cus ||
                          (size_t)(ns * tiles) * g.BM * g.BN * sizeof(float) > work)) break;
            const bool shared = g.BM == 64;
            const double per_cu = (double)(tiles * ns) / num_cus, rounds = std::ceil(per_cu);
            const double load = 0.8 * rounds + 0.2 * per_cu;
            const double t = 2.8 + g.ns * 1e-3 * kper * (shared ? std::max(1.3, load) : load) +
                             g.fix * (shared ? std::max(1.0, per_cu / 2) : rounds) +
                             (ns > 1 ? 1.8 + 0.46 * ns + ns * mn * 8 / 9.2e6 : g.st * c_mb);
            if (t < t_best) {
                t_best = t;
                best = Choice{i, ns};
            }
        }
    }
    return best;
}

template <int I, bool AK, bool BKC, bool EDGE>
static int launch_cfg(hg::Params p, int count, int slices) {
    constexpr HgCfg G = CFG[I];
    p.tiles_m = (p.M + G.BM - 1) / G.BM;
    p.tiles_n = (p.N + G.BN - 1) / G.BN;
    const dim3 block(G.WM * G.WN * 64);
    const unsigned tiles = (unsigned)(p.tiles_m * p.tiles_n);
    if constexpr (EDGE) {
        if (slices > 1 && p.P) {
            p.kper = std::max(((p.K + slices - 1) / slices + KB - 1) / KB * KB, 2 * KB);
            const int ns = (p.K + p.kper - 1) / p.kper;
            hipLaunchKernelGGL((hg::hgemm_kernel<G.BM, G.BN, G.WM, G.WN, KB, G.NS, AK, BKC, G.RA, true, true>),
                               dim3(tiles, (unsigned)ns), block, 0, stream, p);
            G9_HIP(hipGetLastError());
            constexpr int PER = G.BM * G.BN / 512;   // 512 elements of C per wave
            hipLaunchKernelGGL((hg::split_sum<G.BM, G.BN, G.WM, G.WN>), dim3((unsigned)(((long long)tiles * PER + 3) / 4)),
                               dim3(256), 0, stream, p, ns);
            G9_HIP(hipGetLastError());
            return 0;
        }
    }
    hipLaunchKernelGGL((hg::hgemm_kernel<G.BM, G.BN, G.WM, G.WN, KB, G.NS, AK, BKC, G.RA, EDGE>),
                       dim3(tiles, (unsigned)count), block, 0, stream, p);
    G9_HIP(hipGetLastError());
    return 0;
}
template <bool AK, bool BKC>
static int launch_layout(const hg::Params &p, int count, Choice ch, bool whole) {
    if (whole && ch.slices == 1) {
        switch (ch.cfg) {
        case 0: return launch_cfg<0, AK, BKC, false>(p, count, 1);
        case 1: return launch_cfg<1, AK, BKC, false>(p, count, 1);
        case 2: return launch_cfg<2, AK, BKC, false>(p, count, 1);
        }
    }
    switch (ch.cfg) {
    case 0: return launch_cfg<0, AK, BKC, true>(p, count, ch.slices);
    case 1: return launch_cfg<1, AK, BKC, true>(p, count, ch.slices);
    case 2: return launch_cfg<2, AK, BKC, true>(p, count, ch.slices);
    case 5: return launch_cfg<5, AK, BKC, true>(p, count, ch.slices);
    case 6: return launch_cfg<6, AK, BKC, true>(p, count, ch.slices);
    }
    if constexpr (BKC) {
        if (ch.cfg == 3) return launch_cfg<3, AK, BKC, true>(p, count, ch.slices);
    }
    if constexpr (AK) {
        if (ch.cfg == 4) return launch_cfg<4, AK, BKC, true>(p, count, ch.slices);
    }
    G9_FAIL(GEN9BLAS_ERR_UNSUPPORTED, "hgemm: configuration %d for layout A %d B %d", ch.cfg, AK, BKC);
}

}  // namespace hgl

// FP16 products on the direct global→LDS kernel. False, with nothing launched, for those it does not take; otherwise
// *rc is the launch's status.
// The kernel takes operands at 4-byte alignment with even row (and batch) strides, which its direct copies need, and
// more than one k-step of k (exactly one when no operand row ends inside a 16-byte chunk): the k-step it takes through
// registers needs a direct one beside it. Lane offsets inside a tile are 32-bit (lane_span). GEN9BLAS_HGEMM=generic
// forces the general kernel; a forced split-K (GEN9BLAS_SPLITK) leaves it the products that are whole 128×128 tiles.
static bool launch_hgemm_tiles(const GemmCall &c, int *rc) {
    using namespace hgl;
    static const bool generic = [] {
        const char *e = getenv("GEN9BLAS_HGEMM");
        return e && !strcmp(e, "generic");
    }();
    const bool batch = c.count > 1;
    if (generic || c.count > 65535 || c.lda % 2 || c.ldb % 2 || (uintptr_t)c.A % 4 || (uintptr_t)c.B % 4 ||
        (batch && (c.sA % 2 || c.sB % 2)) || std::min(c.lda, c.ldb) < 8)
        return false;
    if (lane_span(!c.tA, c.lda * 2, c.M, KB) >= (1LL << 32) || lane_span(c.tB, c.ldb * 2, c.N, KB) >= (1LL << 32)) return false;
    if (c.K < KB || (c.K == KB && ((c.tA && c.M % 8) || (!c.tB && c.N % 8)))) return false;
    // whole: nothing to check or mask, 16-byte stores
    const auto al16 = [&](const void *x, long long ld, long long s) {
        return (uintptr_t)x % 16 == 0 && ld % 8 == 0 && (!batch || s % 8 == 0);
    };
    const bool aligned = al16(c.A, c.lda, c.sA) && al16(c.B, c.ldb, c.sB) && al16(c.C, c.ldc, c.sC);
    const bool whole128 = aligned && c.M % 128 == 0 && c.N % 128 == 0 && c.K % KB == 0;
    if (splitk_forced() >= 0 && !whole128) return false;
    // the work space of split products is reserved at its bound with the first product here, so that no later call waits
    // for queued work to let it grow
    void *P = nullptr;
    size_t work = 0;
    if (!batch && splitk_forced() < 0) P = splitk_workspace(&work);
    const Choice ch = choose(c, work);
    const HgCfg &g = CFG[ch.cfg];
    if (tiles_of(g, c.M, c.N) > 0x7fffffffLL) return false;
    const bool whole = aligned && c.M % g.BM == 0 && c.N % g.BN == 0 && c.K % KB == 0;

    hg::Params p;
    p.A = reinterpret_cast<const hg::f16 *>(c.A);
    p.B = reinterpret_cast<const hg::f16 *>(c.B);
    p.C = reinterpret_cast<hg::f16 *>(c.C);
    p.lda = c.lda; p.ldb = c.ldb; p.ldc = c.ldc;
    p.sA = batch ? c.sA : 0; p.sB = batch ? c.sB : 0; p.sC = batch ? c.sC : 0;
    p.M = c.M; p.N = c.N; p.K = c.K;
    p.tiles_m = p.tiles_n = 0;
    p.P = reinterpret_cast<float *>(P);
    p.alpha = (float)c.alpha;
    p.beta = (float)c.beta;
    if (c.tA) *rc = c.tB ? launch_layout<false, true>(p, c.count, ch, whole) : launch_layout<false, false>(p, c.count, ch, whole);
    else *rc = c.tB ? launch_layout<true, true>(p, c.count, ch, whole) : launch_layout<true, false>(p, c.count, ch, whole);
    return true;
}

}  // namespace g9
