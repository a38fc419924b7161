// Direct global→LDS copies (global_load_lds_dwordx4) and the waits that go with them, shared by the FP16 and FP32 GEMM
// and the skinny kernels, and 16-byte loads at element alignment. The copies' global addresses need 4-byte alignment
// (a streaming probe on MI355X reads 1 GiB at 6.3-6.4 TB/s at 4-, 8-, 12- and 16-byte alignment alike).
#pragma once
#include <hip/hip_runtime.h>

namespace g9 {

#define G9_LDS __attribute__((address_space(3)))

// One global→LDS copy of 16 bytes per lane: lane L writes LDS bytes lds + 16·L .. +15 with the 16 bytes at
// base + voff (global_load_lds_dwordx4, M0 = LDS address; one wait state between the M0 write and the load).
// Issued by inline assembly: the compiler does not track these writes, so it adds no wait for them before
// unrelated LDS reads. Callers wait for them themselves (wait_vm, and a barrier before other waves read the
// data). Nothing else in the kernels that use it touches M0.
__device__ __forceinline__ void lds_dma16(const void *base, unsigned voff, unsigned lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(base), "s"(lds) : "memory");
}

// s_waitcnt fields (gfx9): vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8; a field at its maximum does not wait.
template <int N> __device__ __forceinline__ void wait_vm() {   // at most N vector-memory loads of this wave in flight
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
__device__ __forceinline__ void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4)); }
// At most s stages of LPS loads each still in flight, s in [0, MAXS].
template <int MAXS, int LPS> __device__ __forceinline__ void wait_vm_stages(int s) {
    if constexpr (MAXS > 0) {
        if (s >= MAXS) { wait_vm<MAXS * LPS>(); return; }
        wait_vm_stages<MAXS - 1, LPS>(s);
    } else {
        wait_vm<0>();
    }
}

typedef unsigned int dma_u32x4 __attribute__((ext_vector_type(4)));

// 16 bytes at an address aligned to the element type only: one global_load_dwordx4 either way (the GPU serves it at
// any element alignment, at the aligned rate when the address is aligned).
template <class T> __device__ __forceinline__ dma_u32x4 load16u(const T *p) {
    typedef T TV __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));
    const TV v = *reinterpret_cast<const TV *>(p);
    return __builtin_bit_cast(dma_u32x4, v);
}

// 16 bytes (V elements) of row r, columns c .. c+V-1 of a row-major matrix X (R valid rows, Cc valid columns, row stride
// ld); zero outside the valid region. In two parts where rows hold at least V elements, so that the loads of all of a
// thread's chunks are on their way before the first is waited for: load16_raw loads the nearest whole chunk inside the
// matrix, one load wherever (r, c) lies, and load16_fix shifts a chunk that crosses the last column into place and clears
// what lies outside.
template <class T> __device__ __forceinline__ dma_u32x4 load16_raw(const T *__restrict__ X, long long ld, int r, int c, int R, int Cc) {
    constexpr int V = 16 / sizeof(T);
    return load16u(X + (long long)min(r, R - 1) * ld + min(c, Cc - V));
}
template <class T> __device__ __forceinline__ dma_u32x4 load16_fix(dma_u32x4 v, int r, int c, int R, int Cc) {
    constexpr int V = 16 / sizeof(T);
    const int bytes = max(c - (Cc - V), 0) * (int)sizeof(T);
    if (bytes & 8) v = dma_u32x4{v[2], v[3], 0, 0};
    if (sizeof(T) < 8 && (bytes & 4)) v = dma_u32x4{v[1], v[2], v[3], 0};
    if (sizeof(T) < 4 && (bytes & 2))
        v = dma_u32x4{v[0] >> 16 | v[1] << 16, v[1] >> 16 | v[2] << 16, v[2] >> 16 | v[3] << 16, v[3] >> 16};
    if (r >= R || c >= Cc) v = dma_u32x4{0, 0, 0, 0};
    return v;
}
// The same for rows of fewer than V elements, one by one.
template <class T> __device__ __forceinline__ dma_u32x4 load16_short(const T *__restrict__ X, long long ld, int r, int c, int R, int Cc) {
    constexpr int V = 16 / sizeof(T);
    union { dma_u32x4 v; T e[V]; } u;
#pragma unroll
    for (int e = 0; e < V; e++) u.e[e] = r < R && c + e < Cc ? X[(long long)r * ld + c + e] : T(0);
    return u.v;
}

}  // namespace g9
