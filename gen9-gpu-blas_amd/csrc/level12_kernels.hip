// Level 1-2 kernels: HBM-streaming, one pass over the operands, FP16 / FP32 / FP64 storage.
//
// Arithmetic follows the reference's level-1/2 kernels (reference: lib/kernels/level12.cl:1-423): FP16 is computed
// in FP32 (R = float for FP16 and FP32, double for FP64); axpy is fma(a, x, y) (level12.cl:133-139); dot / asum / nrm2
// accumulate in FP64 with one partial per workgroup (level12.cl:189-214; the partials are summed here on the device
// in a fixed order instead of on the host); gemv accumulates in R and writes alpha·sum (+ beta·y, y not read when
// beta = 0) (level12.cl:243-423). Vector element i lives at p[o + i·inc] with o = (n-1)·(-inc) for inc < 0, as in
// BLAS. Contiguous, 16-byte-aligned operands move as 16-byte vectors; strided ones element by element.
#include "internal.h"
#include "wave.h"
#include <type_traits>
#include <stdlib.h>

namespace g9 {
namespace l12 {

typedef _Float16 f16;
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef long long ll;

template <class T> struct Comp { using R = float; };
template <> struct Comp<double> { using R = double; };

template <class T> constexpr int VW = 16 / (int)sizeof(T);
template <class T> union Vec {
    u32x4 u;
    T e[VW<T>];
};
template <class T> __device__ __forceinline__ Vec<T> vload(const T *p) {
    Vec<T> v;
    v.u = *reinterpret_cast<const u32x4 *>(p);
    return v;
}
// Streamed operands are read once: nontemporal loads keep them from displacing reusable lines in L2 and MALL (about
// +10 % HBM rate on gfx950 for a single pass). Stores stay ordinary, nontemporal stores measured slower.
template <class T> __device__ __forceinline__ Vec<T> vload_nt(const T *p) {
    Vec<T> v;
    v.u = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p));
    return v;
}
template <class T> __device__ __forceinline__ void vstore(T *p, const Vec<T> &v) { *reinterpret_cast<u32x4 *>(p) = v.u; }
__device__ __forceinline__ float fma_r(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_r(double a, double b, double c) { return __builtin_fma(a, b, c); }

constexpr int NT = 256;
// Grid of a streaming kernel: one 16-byte chunk per thread and grid-stride step, at most `per_cu` blocks per CU
// (4 for kernels with two input streams, 8 for a single read stream: the best HBM rate in a sweep on gfx950).
static unsigned stream_grid(ll chunks, int per_cu = 4) {
    ll g = (chunks + NT - 1) / NT;
    const ll cap = (ll)(num_cus > 0 ? num_cus : 256) * per_cu;
    return (unsigned)(g < 1 ? 1 : g > cap ? cap : g);
}

// ---------------- elementwise: axpy / scal / copy / rot ----------------
// op 0 axpy: y = fma(a, x, y); 1 scal: x = a·x; 2 copy: y = x; 3 rot: x' = h11·x + h12·y, y' = h21·x + h22·y;
// 4 swap.
template <class T, int OP>
__global__ void __launch_bounds__(NT) elem_kernel(int n, typename Comp<T>::R h11, typename Comp<T>::R h12,
                                                  typename Comp<T>::R h21, typename Comp<T>::R h22, T *x, ll ix, T *y,
                                                  ll iy, int vec) {
    using R = typename Comp<T>::R;
    constexpr int V = VW<T>;
    const ll stride = (ll)gridDim.x * NT;
    auto one = [&](T &xe, T &ye) {
        if constexpr (OP == 0) ye = (T)fma_r(h11, (R)xe, (R)ye);
        else if constexpr (OP == 1) xe = (T)(h11 * (R)xe);
        else if constexpr (OP == 2) ye = xe;
        else if constexpr (OP == 3) {
            const R a = (R)xe, b = (R)ye;
            xe = (T)fma_r(h11, a, h12 * b);
            ye = (T)fma_r(h21, a, h22 * b);
        } else {
            const T t = xe;
            xe = ye;
            ye = t;
        }
    };
    if (vec) {
        const ll nv = n / V;
        for (ll c = (ll)blockIdx.x * NT + threadIdx.x; c < nv; c += stride) {
            Vec<T> xv, yv;
            xv = vload_nt(x + c * V);
            if constexpr (OP == 0 || OP >= 3) yv = vload_nt(y + c * V);
#pragma unroll
            for (int e = 0; e < V; e++) one(xv.e[e], yv.e[e]);
            if constexpr (OP == 1 || OP >= 3) vstore(x + c * V, xv);
            if constexpr (OP == 0 || OP == 2 || OP >= 3) vstore(y + c * V, yv);
        }
        for (ll i = nv * V + (ll)blockIdx.x * NT + threadIdx.x; i < n; i += stride) {
            T dummy = T(0);
            one(x[i], OP == 1 ? dummy : y[i]);
        }
        return;
    }
    for (ll i = (ll)blockIdx.x * NT + threadIdx.x; i < n; i += stride) {
        T dummy = T(0);
        one(x[i * ix], OP == 1 ? dummy : y[i * iy]);
    }
}

// ---------------- reductions (FP64) ----------------
__device__ __forceinline__ double wave_sum(double s) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) s += __shfl_xor(s, d);
    return s;
}
__device__ __forceinline__ double block_sum(double s) {
    __shared__ double ws[NT / 64];
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = s;
    __syncthreads();
    double t = 0;
    if (threadIdx.x == 0)
#pragma unroll
        for (int w = 0; w < NT / 64; w++) t += ws[w];
    return t;   // valid in thread 0
}

// Two kernels: every block writes its FP64 partial, then reduce_final adds the partials in index order, so the
// result does not depend on block scheduling. (Finishing in the last block instead needs a device-scope fence per
// block, which writes back and invalidates the L2 of the XCD: about 35 % of the HBM rate at 1 GiB on gfx950.)
// A single block's partial is the result itself (square root taken for nrm2) and goes to `part` without the second
// kernel.
template <class T, int MODE>
__global__ void __launch_bounds__(NT) reduce_kernel(int n, const T *x, ll ix, const T *y, ll iy, int vec, double *part) {
    constexpr int V = VW<T>;
    const ll stride = (ll)gridDim.x * NT;
    double s0 = 0, s1 = 0;   // two chains: FP64 fma latency does not serialize the stream
    auto acc = [&](double &s, double a, double b) {
        if constexpr (MODE == 0) s = __builtin_fma(a, b, s);
        else if constexpr (MODE == 1) s += __builtin_fabs(a);
        else s = __builtin_fma(a, a, s);
    };
    ll tail = 0;
    if (vec) {
        // Each step a block reads U·NT consecutive chunks (16 KiB for FP32 asum) with every load issued before the
        // first add: 4 loads of 16 bytes in flight per lane (dot: 2 of x and 2 of y), and the blocks in flight cover
        // one contiguous span of memory.
        constexpr int U = MODE == 0 ? 2 : 4;
        const ll nv = n / V, big = (ll)U * NT, nsc = nv / big;
        for (ll sc = blockIdx.x; sc < nsc; sc += gridDim.x) {
            const ll c0 = sc * big + threadIdx.x;
            Vec<T> xv[U], yv[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                xv[u] = vload_nt(x + (c0 + u * NT) * V);
                if constexpr (MODE == 0) yv[u] = vload_nt(y + (c0 + u * NT) * V);
            }
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int e = 0; e < V; e++)
                    acc(e & 1 ? s1 : s0, (double)xv[u].e[e], MODE == 0 ? (double)yv[u].e[e] : 0.0);
        }
        ll c = nsc * big + (ll)blockIdx.x * NT + threadIdx.x;   // the chunks past the last whole super-chunk
        for (; c < nv; c += stride) {
            const Vec<T> xv = vload_nt(x + c * V);
            Vec<T> yv;
            if constexpr (MODE == 0) yv = vload_nt(y + c * V);
#pragma unroll
            for (int e = 0; e < V; e++) acc(e & 1 ? s1 : s0, (double)xv.e[e], MODE == 0 ? (double)yv.e[e] : 0.0);
        }
        tail = nv * V;
        ix = 1;
        iy = 1;
    }
    for (ll i = tail + (ll)blockIdx.x * NT + threadIdx.x; i < n; i += stride)
        acc(s0, (double)x[i * ix], MODE == 0 ? (double)y[i * iy] : 0.0);
    const double t = block_sum(s0 + s1);
    if (threadIdx.x == 0) part[blockIdx.x] = MODE == 2 && gridDim.x == 1 ? __builtin_sqrt(t) : t;
}

// Sum of np ≤ FIN·NT partials (more are handled by the plain loop): all loads are issued before the first add, so
// the kernel costs about one memory latency.
constexpr int FIN = 8;
__global__ void __launch_bounds__(NT) reduce_final(int np, const double *part, int mode, double *out) {
    double v[FIN];
#pragma unroll
    for (int j = 0; j < FIN; j++) {
        const int i = threadIdx.x + j * NT;
        v[j] = i < np ? part[i] : 0.0;
    }
    double s = 0;
#pragma unroll
    for (int j = 0; j < FIN; j++) s += v[j];
    for (int i = threadIdx.x + FIN * NT; i < np; i += NT) s += part[i];
    const double t = block_sum(s);
    if (threadIdx.x == 0) *out = mode == 2 ? __builtin_sqrt(t) : t;
}

// ---------------- iamax: first index of the largest |x|; NaN skipped, all NaN (or n = 0 in a part) → index 0 ----------------
struct ValIdx {
    double v;
    long long i;
};
__device__ __forceinline__ ValIdx better(ValIdx a, ValIdx b) {
    return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}
__device__ __forceinline__ ValIdx block_best(ValIdx b) {
    __shared__ double sv[NT];
    __shared__ long long si[NT];
    sv[threadIdx.x] = b.v;
    si[threadIdx.x] = b.i;
    __syncthreads();
    for (int d = NT / 2; d >= 1; d >>= 1) {
        if ((int)threadIdx.x < d) {
            const ValIdx o = better(ValIdx{sv[threadIdx.x], si[threadIdx.x]}, ValIdx{sv[threadIdx.x + d], si[threadIdx.x + d]});
            sv[threadIdx.x] = o.v;
            si[threadIdx.x] = o.i;
        }
        __syncthreads();
    }
    return ValIdx{sv[0], si[0]};
}
template <class T>
__global__ void __launch_bounds__(NT) iamax_kernel(int n, const T *x, ll ix, double *pv, long long *pi) {
    ValIdx b{-1.0, 0x7fffffffffffffffLL};
    for (ll i = (ll)blockIdx.x * NT + threadIdx.x; i < n; i += (ll)gridDim.x * NT) {
        const double a = __builtin_fabs((double)x[i * ix]);
        if (a == a) b = better(b, ValIdx{a, i});   // a != a: NaN, skipped
    }
    b = block_best(b);
    if (threadIdx.x == 0) {
        pv[blockIdx.x] = b.v;
        pi[blockIdx.x] = b.i;
    }
}
__global__ void __launch_bounds__(NT) iamax_final(int np, const double *pv, const long long *pi, long long *out) {
    ValIdx b{-1.0, 0x7fffffffffffffffLL};
    for (int i = threadIdx.x; i < np; i += NT) b = better(b, ValIdx{pv[i], pi[i]});
    b = block_best(b);
    if (threadIdx.x == 0) *out = b.i == 0x7fffffffffffffffLL ? 0 : b.i;
}

// ---------------- GEMV ----------------
// Both directions read A once, 16 bytes per lane, at whatever alignment its rows have (an odd row length or a
// submatrix leaves rows aligned to their elements only; the GPU serves such loads), and are bound by the bytes they
// keep in flight: every batch of loads, the last partial one included, is issued before its first product.
template <int ES> struct Unaligned;
template <> struct Unaligned<2> { typedef u32x4 type __attribute__((aligned(2))); };
template <> struct Unaligned<4> { typedef u32x4 type __attribute__((aligned(4))); };
template <> struct Unaligned<8> { typedef u32x4 type __attribute__((aligned(8))); };
// NTL: nontemporal, for an A too large to be found in the last-level cache by the next product with it.
template <bool NTL, class T> __device__ __forceinline__ Vec<T> vload_a(const T *p) {
    Vec<T> v;
    const auto *q = reinterpret_cast<const typename Unaligned<(int)sizeof(T)>::type *>(p);
    if constexpr (NTL) v.u = __builtin_nontemporal_load(q);
    else v.u = *q;
    return v;
}
// No-trans, y = alpha·A·x + beta·y: RWN rows per group of KS waves, whose lanes stream 16 bytes of each row per step
// (1 KiB per row and wave, steps dealt to the waves in turn) and reuse each chunk of x for the RWN rows. The RWN sums
// are reduced across the wave by the transposing butterfly, the KS waves' sums added in LDS in wave order. U steps per
// batch. VEC false: an element per lane and step, for short FP16 rows, which would leave most lanes of a 16-byte step idle,
// and for an x with a stride, whose elements the lanes then load side by side.
// MI355X, µs per call, FP32 unless said; before the 16-byte loads at element alignment (element-wise loads for rows not
// 16-byte aligned, 16 rows per block throughout) -> now: 6000×1501 10.3 -> 5.8, 6000×1500 6.5 -> 5.8, 1000×8192 13.5 -> 5.3,
// 300×40000 75 -> 12, 16384×16383 188 -> 168, FP16 8191×4097 23.2 -> 11.3.
constexpr int RWN = 4;
template <class T, bool VEC, bool NTL, int KS, int U>
__global__ void __launch_bounds__(NT) gemv_n_kernel(int M, int N, typename Comp<T>::R alpha, const T *A, ll lda, const T *x,
                                                    ll ix, typename Comp<T>::R beta, T *y, ll iy) {
    static_assert(KS == 1 || KS == NT / 64, "rows of a wave, or of a block");
    using R = typename Comp<T>::R;
    constexpr int V = VEC ? VW<T> : 1, SW = KS * 64 * V;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r0 = (KS == 1 ? (int)blockIdx.x * (NT / 64) + w : (int)blockIdx.x) * RWN, kw = KS == 1 ? 0 : w;
    if (KS == 1 && r0 >= M) return;
    const T *ar[RWN];
#pragma unroll
    for (int r = 0; r < RWN; r++) ar[r] = A + (ll)min(r0 + r, M - 1) * lda;
    R s[RWN];
#pragma unroll
    for (int r = 0; r < RWN; r++) s[r] = 0;
    if constexpr (VEC) {
        const int nvec = N - N % V;
        // US steps from column j0 of this wave; LAST: lanes past nvec in the last of them load nothing and add zeros
        auto batch = [&](int j0, auto us, auto last) {
            constexpr int US = decltype(us)::value;
            constexpr bool LAST = decltype(last)::value;
            Vec<T> xv[US], av[US][RWN];
#pragma unroll
            for (int u = 0; u < US; u++) {
                const unsigned j = (unsigned)j0 + u * SW + lane * V;
                const auto load = [&] {
                    xv[u].u = *reinterpret_cast<const typename Unaligned<(int)sizeof(T)>::type *>(x + j);
#pragma unroll
                    for (int r = 0; r < RWN; r++) av[u][r] = vload_a<NTL>(ar[r] + j);
                };
                if (LAST && u == US - 1) {
                    xv[u].u = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
                    for (int r = 0; r < RWN; r++) av[u][r].u = u32x4{0u, 0u, 0u, 0u};
                    if (j < (unsigned)nvec) load();
                } else {
                    load();
                }
            }
#pragma unroll
            for (int u = 0; u < US; u++)
#pragma unroll
                for (int r = 0; r < RWN; r++)
#pragma unroll
                    for (int e = 0; e < V; e++) s[r] = fma_r((R)av[u][r].e[e], (R)xv[u].e[e], s[r]);
        };
        using No = std::false_type;
        using Yes = std::true_type;
        int j0 = kw * 64 * V;
        for (; nvec - j0 >= U * SW; j0 += U * SW) batch(j0, std::integral_constant<int, U>(), No());
        // the columns past the last whole 16 bytes, one per lane of the first wave, loaded ahead of the last batch
        const bool tail = kw == 0 && nvec + lane < N;
        R at[RWN], xt = 0;
#pragma unroll
        for (int r = 0; r < RWN; r++) at[r] = 0;
        if (tail) {
            xt = (R)x[nvec + lane];
#pragma unroll
            for (int r = 0; r < RWN; r++) at[r] = (R)ar[r][nvec + lane];
        }
        const int left = j0 < nvec ? (nvec - j0 + SW - 1) / SW : 0;   // steps of this wave still to do, 0 .. U
        if constexpr (U > 2) {
            if (left == 4) batch(j0, std::integral_constant<int, 4>(), Yes());
            else if (left == 3) batch(j0, std::integral_constant<int, 3>(), Yes());
        }
        if (left == 2) batch(j0, std::integral_constant<int, 2>(), Yes());
        else if (left == 1) batch(j0, std::integral_constant<int, 1>(), Yes());
        if (tail)
#pragma unroll
            for (int r = 0; r < RWN; r++) s[r] = fma_r(at[r], xt, s[r]);
    } else {
        ll j = kw * 64 + lane;
        for (; j + (U - 1) * SW < N; j += U * SW) {
            T xv[U], av[U][RWN];
#pragma unroll
            for (int u = 0; u < U; u++) {
                xv[u] = x[(j + u * SW) * ix];
#pragma unroll
                for (int r = 0; r < RWN; r++) av[u][r] = ar[r][j + u * SW];
            }
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int r = 0; r < RWN; r++) s[r] = fma_r((R)av[u][r], (R)xv[u], s[r]);
        }
        for (; j < N; j += SW) {
            const R xj = (R)x[j * ix];
#pragma unroll
            for (int r = 0; r < RWN; r++) s[r] = fma_r((R)ar[r][j], xj, s[r]);
        }
    }
    // butterfly over the RWN row sums: two halving exchanges, then plain sums
    int base = 0;
    butterfly<0, RWN>(s, lane, base);
    R sum = s[0];
    int row = r0 + base;
    bool writer = (lane & (64 / RWN - 1)) == 0;
    if constexpr (KS > 1) {
        __shared__ R red[KS][RWN];
        if (writer) red[w][base] = sum;
        __syncthreads();
        writer = threadIdx.x < RWN;
        if (writer) {
            row = r0 + (int)threadIdx.x;
            sum = red[0][threadIdx.x];
#pragma unroll
            for (int q = 1; q < KS; q++) sum += red[q][threadIdx.x];
        }
    }
    if (writer && row < M) {
        T *yp = y + (ll)row * iy;
        *yp = (T)(beta == R(0) ? alpha * sum : fma_r(alpha, sum, beta * (R)*yp));
    }
}

// Trans, y = alpha·Aᵀ·x + beta·y, at most FEW rows: a thread owns V columns (16 bytes per lane) and all the rows, in four
// groups whose sums are added in order, as the waves of the kernel below would. Those would have a row or two each, and a
// pass through LDS after it: MI355X, µs, FP64 × 1000000 columns, 1 row 7.6 -> 5.8, 4 rows 12.5 -> 6.1, FP32 4 rows 7.7 -> 4.7
// (16 rows: FP16 8.6 against 6.9).
constexpr int FEW = 8;
template <class T>
__global__ void __launch_bounds__(NT) gemv_t_few_kernel(int M, int N, const T *A, ll lda, const T *x, ll ix,
                                                        typename Comp<T>::R alpha, typename Comp<T>::R beta, T *y, ll iy) {
    using R = typename Comp<T>::R;
    constexpr int V = VW<T>, G = FEW / 4;   // rows of a group
    const ll cb = ((ll)blockIdx.x * NT + threadIdx.x) * V;
    if (cb >= N) return;
    const int c0 = (int)max(min(cb, (ll)N - V), 0ll);   // as below: the last thread's columns end with the row
    const int rw = (M + 3) / 4;
    Vec<T> av[FEW];
    R xv[FEW];
    const auto row = [&](int u) { return min(u / G * rw + min(u % G, rw - 1), M - 1); };
    if (N >= V) {
#pragma unroll
        for (int u = 0; u < FEW; u++) av[u] = vload_a<false>(A + row(u) * lda + c0);
    } else {
#pragma unroll
        for (int u = 0; u < FEW; u++)
#pragma unroll
            for (int e = 0; e < V; e++) av[u].e[e] = A[row(u) * lda + min(e, N - 1)];
    }
#pragma unroll
    for (int u = 0; u < FEW; u++) xv[u] = (R)x[row(u) * ix];
    R s[V];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        R t[V];
#pragma unroll
        for (int e = 0; e < V; e++) t[e] = 0;
#pragma unroll
        for (int u = 0; u < G; u++)
            if (u < rw && q * rw + u < M)
#pragma unroll
                for (int e = 0; e < V; e++) t[e] = fma_r((R)av[q * G + u].e[e], xv[q * G + u], t[e]);
#pragma unroll
        for (int e = 0; e < V; e++) s[e] = q == 0 ? t[e] : s[e] + t[e];
    }
#pragma unroll
    for (int e = 0; e < V; e++)
        if (c0 + e >= cb && c0 + e < N) {
            T *yp = y + (c0 + e) * iy;
            *yp = (T)(beta == R(0) ? alpha * s[e] : fma_r(alpha, s[e], beta * (R)*yp));
        }
}

// Trans, y = alpha·Aᵀ·x + beta·y. Stage 1: a block owns 64·V columns (16 bytes per lane) and a band of rpp rows, a
// quarter of it per wave; the waves' sums are added in LDS in wave order and go to P[part][col]. Stage 2: y[col] =
// alpha·Σ_part P[part][col] + beta·y[col] in a fixed order. With one part stage 1 writes y. The last lane's columns
// that would pass the row's end start V before it; the ones another lane owns are summed and not written. The sum over
// a block's waves quarters the partials that stage 2 reads.
// MI355X, µs per call with stage 2, FP32 unless said, before (element-wise loads for rows not 16-byte aligned, 1024
// columns and one partial per block row band) -> now: 6000×1501 23.9 -> 10.2, 6000×1500 15.2 -> 10.0, 40000×333 49.8 ->
// 15.6, 16384×16383 446 -> 179, FP16 8191×4097 47.7 -> 16; 16384×8192 84.6 -> 82.5.
template <class T, bool NTL>
__global__ void __launch_bounds__(NT) gemv_t1_kernel(int M, int N, int rpp, const T *A, ll lda, const T *x, ll ix,
                                                     typename Comp<T>::R *P, int direct, typename Comp<T>::R alpha,
                                                     typename Comp<T>::R beta, T *y, ll iy) {
    using R = typename Comp<T>::R;
    constexpr int V = VW<T>, W = NT / 64, U = 8;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int b0 = blockIdx.x * 64 * V, cb = b0 + lane * V, c0 = max(min(cb, N - V), 0);
    const int part = blockIdx.y, i0 = part * rpp, i1 = min(M, i0 + rpp), rw = (i1 - i0 + W - 1) / W;
    int i = i0 + w * rw;
    const int a1 = min(i1, i + rw);
    R s[V];
#pragma unroll
    for (int e = 0; e < V; e++) s[e] = 0;
    if (N >= V) {
        const T *Ac = A + c0;
        // U rows per step, their loads all issued before the first product
        for (; i + U <= a1; i += U) {
            Vec<T> av[U];
            R xv[U];
#pragma unroll
            for (int u = 0; u < U; u++) av[u] = vload_a<NTL>(Ac + (ll)(i + u) * lda);
#pragma unroll
            for (int u = 0; u < U; u++) xv[u] = (R)x[(ll)(i + u) * ix];
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int e = 0; e < V; e++) s[e] = fma_r((R)av[u].e[e], xv[u], s[e]);
        }
        if (i < a1) {   // the last rows, fewer than U
            Vec<T> av[U - 1];
            R xv[U - 1];
#pragma unroll
            for (int u = 0; u < U - 1; u++) av[u] = vload_a<NTL>(Ac + (ll)min(i + u, a1 - 1) * lda);
#pragma unroll
            for (int u = 0; u < U - 1; u++) xv[u] = (R)x[(ll)min(i + u, a1 - 1) * ix];
#pragma unroll
            for (int u = 0; u < U - 1; u++)
                if (i + u < a1)
#pragma unroll
                    for (int e = 0; e < V; e++) s[e] = fma_r((R)av[u].e[e], xv[u], s[e]);
        }
    } else {
        for (; i < a1; i++) {
            const R xv = (R)x[(ll)i * ix];
#pragma unroll
            for (int e = 0; e < V; e++) s[e] = fma_r((R)A[(ll)i * lda + min(e, N - 1)], xv, s[e]);
        }
    }
    __shared__ R red[W][64 * V];
#pragma unroll
    for (int e = 0; e < V; e++)
        if (c0 + e >= cb) red[w][c0 + e - b0] = s[e];
    __syncthreads();
    for (int t = threadIdx.x; t < 64 * V && b0 + t < N; t += NT) {
        R sum = red[0][t];
#pragma unroll
        for (int q = 1; q < W; q++) sum += red[q][t];
        if (direct) {
            T *yp = y + (ll)(b0 + t) * iy;
            *yp = (T)(beta == R(0) ? alpha * sum : fma_r(alpha, sum, beta * (R)*yp));
        } else {
            P[(ll)part * N + b0 + t] = sum;
        }
    }
}
// 64 columns per block; the block's G waves each sum every G-th part (loads issued 8 at a time, added in part order),
// then wave 0 adds the G sums in wave order: a fixed summation order for every column.
template <class T, int G>
__global__ void __launch_bounds__(G * 64) gemv_t2_kernel(int N, int parts, const typename Comp<T>::R *P,
                                                     typename Comp<T>::R alpha, typename Comp<T>::R beta, T *y, ll iy) {
    using R = typename Comp<T>::R;
    const int j = blockIdx.x * 64 + (threadIdx.x & 63), jc = min(j, N - 1);
    const int gq = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    R t = 0;
    for (int r = gq; r < parts; r += 8 * G) {
        R v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = P[(ll)min(r + u * G, parts - 1) * N + jc];
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (r + u * G < parts) t += v[u];
    }
    __shared__ R red[G][64];
    red[gq][threadIdx.x & 63] = t;
    __syncthreads();
    if (gq == 0 && j < N) {
        R sum = red[0][threadIdx.x];
#pragma unroll
        for (int q = 1; q < G; q++) sum += red[q][threadIdx.x];
        T *yp = y + (ll)j * iy;
        *yp = (T)(beta == R(0) ? alpha * sum : fma_r(alpha, sum, beta * (R)*yp));
    }
}

// ---------------- GER: A = alpha·x·yᵀ + A ----------------
template <class T>
__global__ void __launch_bounds__(NT) ger_kernel(int M, int N, typename Comp<T>::R alpha, const T *x, ll ix, const T *y,
                                                 ll iy, T *A, ll lda) {
    using R = typename Comp<T>::R;
    const int i = blockIdx.y;
    const R ax = alpha * (R)x[(ll)i * ix];
    for (int j = blockIdx.x * NT + threadIdx.x; j < N; j += gridDim.x * NT) {
        T *a = A + (ll)i * lda + j;
        *a = (T)fma_r(ax, (R)y[(ll)j * iy], (R)*a);
    }
}

}  // namespace l12

using namespace l12;

// ---------------- launchers ----------------
template <class F> static int by_type(int es, F f) {
    if (es == 2) return f((f16 *)nullptr);
    if (es == 4) return f((float *)nullptr);
    return f((double *)nullptr);
}
static bool al16(const void *p) { return (uintptr_t)p % 16 == 0; }

template <int OP>
static int elem(int es, int n, double h11, double h12, double h21, double h22, void *x, ll ox, ll ix, void *y, ll oy, ll iy) {
    return by_type(es, [&](auto *tag) -> int {
        using T = std::remove_pointer_t<decltype(tag)>;
        using R = typename Comp<T>::R;
        T *xp = (T *)x + ox, *yp = y ? (T *)y + oy : nullptr;
        const bool vec = ix == 1 && (OP == 1 || iy == 1) && al16(xp) && (OP == 1 || al16(yp));
        const unsigned g = stream_grid(vec ? (n + VW<T> - 1) / VW<T> : n);
        hipLaunchKernelGGL((elem_kernel<T, OP>), dim3(g), dim3(NT), 0, stream, n, (R)h11, (R)h12, (R)h21, (R)h22, xp, ix,
                           yp, iy, (int)vec);
        G9_HIP(hipGetLastError());
        return 0;
    });
}

int launch_axpy(int es, int n, double a, const void *x, ll ox, ll ix, void *y, ll oy, ll iy) {
    return elem<0>(es, n, a, 0, 0, 0, const_cast<void *>(x), ox, ix, y, oy, iy);
}
int launch_scal(int es, int n, double a, void *x, ll ox, ll ix) { return elem<1>(es, n, a, 0, 0, 0, x, ox, ix, nullptr, 0, 1); }
int launch_copy(int es, int n, const void *x, ll ox, ll ix, void *y, ll oy, ll iy) {
    return elem<2>(es, n, 0, 0, 0, 0, const_cast<void *>(x), ox, ix, y, oy, iy);
}
int launch_rot(int es, int n, void *x, ll ox, ll ix, void *y, ll oy, ll iy, double h11, double h12, double h21, double h22,
               int swap) {
    if (swap) return elem<4>(es, n, 0, 0, 0, 0, x, ox, ix, y, oy, iy);
    return elem<3>(es, n, h11, h12, h21, h22, x, ox, ix, y, oy, iy);
}

// Reductions of up to one step of one block (1024 chunks) run as that block alone: the second kernel's launch costs more
// than the other CUs save (nrm2 of 1501 FP32 values, with the wait for the result: 14.8 -> 11.8 µs).
constexpr ll REDUCE_ONE = 4 * NT;
int launch_reduce(int es, int mode, int n, const void *x, ll ox, ll ix, const void *y, ll oy, ll iy, double *result) {
    return by_type(es, [&](auto *tag) -> int {
        using T = std::remove_pointer_t<decltype(tag)>;
        const T *xp = (const T *)x + ox, *yp = y ? (const T *)y + oy : xp;
        const bool vec = ix == 1 && (mode != 0 || iy == 1) && al16(xp) && (mode != 0 || al16(yp));
        const ll chunks = vec ? (n + VW<T> - 1) / VW<T> : n;
        const unsigned g = chunks <= REDUCE_ONE ? 1u : stream_grid(chunks, mode == 0 ? 4 : 8);
        double *part = result;
        if (g > 1) {
            void *pp;
            G9_TRY(scratch(SLOT_P, g * sizeof(double), &pp));
            part = (double *)pp;
        }
        if (mode == 0) hipLaunchKernelGGL((reduce_kernel<T, 0>), dim3(g), dim3(NT), 0, stream, n, xp, ix, yp, iy, (int)vec, part);
        else if (mode == 1) hipLaunchKernelGGL((reduce_kernel<T, 1>), dim3(g), dim3(NT), 0, stream, n, xp, ix, yp, iy, (int)vec, part);
        else hipLaunchKernelGGL((reduce_kernel<T, 2>), dim3(g), dim3(NT), 0, stream, n, xp, ix, yp, iy, (int)vec, part);
        G9_HIP(hipGetLastError());
        if (g > 1) {
            hipLaunchKernelGGL(reduce_final, dim3(1), dim3(NT), 0, stream, (int)g, (const double *)part, mode, result);
            G9_HIP(hipGetLastError());
        }
        return 0;
    });
}

int launch_iamax(int es, int n, const void *x, ll ox, ll ix, long long *result) {
    return by_type(es, [&](auto *tag) -> int {
        using T = std::remove_pointer_t<decltype(tag)>;
        const T *xp = (const T *)x + ox;
        const unsigned g = stream_grid(n);
        void *pp;
        G9_TRY(scratch(SLOT_P, g * (sizeof(double) + sizeof(long long)), &pp));
        double *pv = (double *)pp;
        long long *pi = (long long *)(pv + g);
        hipLaunchKernelGGL((iamax_kernel<T>), dim3(g), dim3(NT), 0, stream, n, xp, ix, pv, pi);
        G9_HIP(hipGetLastError());
        hipLaunchKernelGGL(iamax_final, dim3(1), dim3(NT), 0, stream, (int)g, (const double *)pv, (const long long *)pi,
                           result);
        G9_HIP(hipGetLastError());
        return 0;
    });
}

constexpr int GEMV_T_PER_CU = 3;
int launch_gemv(int es, int trans, int M, int N, double alpha, const void *A, ll lda, const void *x, ll ox, ll ix,
                double beta, void *y, ll oy, ll iy) {
    return by_type(es, [&](auto *tag) -> int {
        using T = std::remove_pointer_t<decltype(tag)>;
        using R = typename Comp<T>::R;
        const T *Ap = (const T *)A, *xp = (const T *)x + ox;
        T *yp = (T *)y + oy;
        // A of more than the 256 MiB last-level cache is read past it (nontemporal); a smaller one, which a solver's next
        // product with it finds there, is not. No-trans, µs, nontemporal against plain loads: FP32 16384×8192 (512 MiB) 104
        // against 122, 32768×4096 92 against 113; FP64 16384×2048 (256 MiB) 47 against 40.
        const bool ntl = (double)M * (double)N * sizeof(T) > (double)(256 << 20);
        if (!trans) {
            // An element per lane: FP16 rows of at most 128 of them (100000×100 6.1 µs against 7.9, ×200 10.2 against 8.1;
            // FP32 and FP64 rows of up to 64 take 5.4 against 6.2, but their products then round before they are added:
            // 1000×50 7.1e-8 of the result against 6.2e-8), and an x with a stride, where rows are not long nor A large:
            // those have x gathered first. FP16 16384×4096 25 µs (loads of x inside each lane's 16 bytes instead 39), 8192²
            // gathered 23 (36).
            bool vec = sizeof(T) > 2 || N > 128;
            if (vec && ix != 1) {
                void *g = nullptr;
                vec = (ntl || N > 2048 * (int)sizeof(T)) && (g = try_scratch(SLOT_P, (size_t)N * sizeof(T)));
                if (vec) {
                    G9_TRY(launch_copy(es, N, x, ox, ix, g, 0, 1));
                    xp = (const T *)g;
                    ix = 1;
                }
            }
            // The four waves of a block share its rows where rows alone would leave CUs with few waves (fewer than 4
            // blocks per CU), unless a row is so short that they would have nothing to share.
            const unsigned g = (unsigned)((M + RWN * (NT / 64) - 1) / (RWN * (NT / 64)));
            const bool share = g < 4u * (unsigned)num_cus && N > 2 * 64 * (vec ? VW<T> : 1);
            // Batches of four steps where a row holds four of them, else of two, whose registers leave more waves: FP16
            // 16384×2048 11.5 against 13.8, FP32 32768×4096 92 against 101, FP64 40000×3000 137 against 146; FP32 100000×200
            // (one step) 14.8 against 12.7, 4096² (shared rows, from the cache) 12.4 against 11.2.
            const bool four = (!share || ntl) && N >= 4 * 64 * VW<T> * (share ? NT / 64 : 1);
            const auto go = [&](auto vc, auto nt, auto us) {
                constexpr bool VEC = decltype(vc)::value, NTL = decltype(nt)::value;
                constexpr int U = decltype(us)::value;
                const auto kern = share ? gemv_n_kernel<T, VEC, NTL, NT / 64, U> : gemv_n_kernel<T, VEC, NTL, 1, U>;
                hipLaunchKernelGGL(kern, dim3(share ? (unsigned)((M + RWN - 1) / RWN) : g), dim3(NT), 0, stream, M, N, (R)alpha,
                                   Ap, lda, xp, ix, (R)beta, yp, iy);
            };
            using Yes = std::true_type;
            using No = std::false_type;
            using One = std::integral_constant<int, 1>;   // element-wise: waves enough hide a step's loads
            using Two = std::integral_constant<int, 2>;
            using Four = std::integral_constant<int, 4>;
            if (!vec) share ? go(No(), No(), Four()) : go(No(), No(), One());
            else if (four) ntl ? go(Yes(), Yes(), Four()) : go(Yes(), No(), Four());
            else ntl ? go(Yes(), Yes(), Two()) : go(Yes(), No(), Two());
            G9_HIP(hipGetLastError());
            return 0;
        }
        if (M <= FEW) {
            hipLaunchKernelGGL((gemv_t_few_kernel<T>), dim3((unsigned)(((ll)N + NT * VW<T> - 1) / (NT * VW<T>))), dim3(NT), 0,
                               stream, M, N, Ap, lda, xp, ix, (R)alpha, (R)beta, yp, iy);
            G9_HIP(hipGetLastError());
            return 0;
        }
        constexpr int V = VW<T>, W = NT / 64;
        const int cblocks = (N + 64 * V - 1) / (64 * V);
        // about GEMV_T_PER_CU blocks per CU, each summing a band of rows into FP32 (FP64) partials; whole batches of 8
        // rows per wave
        const int tgt = GEMV_T_PER_CU * (num_cus > 0 ? num_cus : 256);
        int parts = (tgt + cblocks - 1) / cblocks;
        const int maxparts = (M + 8 * W - 1) / (8 * W);
        if (parts > maxparts) parts = maxparts;
        if (parts < 1) parts = 1;
        const int rpp = (int)(((ll)M + (ll)parts * 8 * W - 1) / ((ll)parts * 8 * W)) * 8 * W;
        parts = (int)(((ll)M + rpp - 1) / rpp);
        R *P = nullptr;
        if (parts > 1) {
            void *pp;
            G9_TRY(scratch(SLOT_P, (size_t)parts * N * sizeof(R), &pp));
            P = (R *)pp;
        }
        const dim3 grid((unsigned)cblocks, (unsigned)parts);
        hipLaunchKernelGGL((ntl ? gemv_t1_kernel<T, true> : gemv_t1_kernel<T, false>), grid, dim3(NT), 0, stream, M, N, rpp, Ap, lda, xp, ix, P, (int)(parts == 1), (R)alpha, (R)beta, yp, iy);
        G9_HIP(hipGetLastError());
        if (parts > 1) {
            const dim3 g2((unsigned)((N + 63) / 64));
            if (parts > 32) hipLaunchKernelGGL((gemv_t2_kernel<T, 16>), g2, dim3(1024), 0, stream, N, parts, (const R *)P, (R)alpha, (R)beta, yp, iy);
            else hipLaunchKernelGGL((gemv_t2_kernel<T, 4>), g2, dim3(256), 0, stream, N, parts, (const R *)P, (R)alpha, (R)beta, yp, iy);
            G9_HIP(hipGetLastError());
        }
        return 0;
    });
}

int launch_ger(int es, int M, int N, double alpha, const void *x, ll ox, ll ix, const void *y, ll oy, ll iy, void *A, ll lda) {
    return by_type(es, [&](auto *tag) -> int {
        using T = std::remove_pointer_t<decltype(tag)>;
        using R = typename Comp<T>::R;
        if (M > 65535) G9_FAIL(GEN9BLAS_ERR_UNSUPPORTED, "ger: M = %d > 65535", M);
        const unsigned gx = (unsigned)((N + NT - 1) / NT < 64 ? (N + NT - 1) / NT : 64);
        hipLaunchKernelGGL((ger_kernel<T>), dim3(gx, (unsigned)M), dim3(NT), 0, stream, M, N, (R)alpha, (const T *)x + ox, ix,
                           (const T *)y + oy, iy, (T *)A, lda);
        G9_HIP(hipGetLastError());
        return 0;
    });
}

}  // namespace g9
