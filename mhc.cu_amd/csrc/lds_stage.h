// Pieces of the kernels that keep global memory busy across barriers (bwd_slab.hip, bwd_slab8.hip, bwd_static.hip): loads from global memory straight into LDS, waits and
// barriers that count them, and the order of the chunks of a row there.
#pragma once
#include "mhc_common.h"

namespace mhc {

// global -> LDS without registers in between: lane i's BYTES from base + off to lds + i * BYTES.  As assembly because the
// compiler would wait for ALL of them before the next LDS access of any kind; the loaders wait by count (wait_vmem).
// M0 is used by nothing else here (LDS instructions of this architecture do not read it).
template <int BYTES> __device__ __forceinline__ void load_to_lds(const void *base, uint32_t off, uint32_t lds) {
    static_assert(BYTES == 4 || BYTES == 16, "one or four words per lane");
    const uint64_t p = (uint64_t)(uintptr_t)base;
    if constexpr (BYTES == 16) asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(p), "s"(lds) : "memory");
    else asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(off), "s"(p), "s"(lds) : "memory");
}
__device__ __forceinline__ uint32_t lds_address(const void *p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char *)p;
}
template <int K> __device__ __forceinline__ void wait_vmem() {  // at most K younger vector memory operations in flight
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(K) : "memory");
}
// Barrier of the whole workgroup that waits for this wave's LDS accesses but not for its global ones (__syncthreads
// is free to wait for both).
__device__ __forceinline__ void stage_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// K floats from LDS, 16 bytes at a time where they are whole 16-byte pieces (and then aligned to them).
template <int K> __device__ __forceinline__ void lds_floats(const float *p, float *v) {
    if constexpr (K % 4 == 0) {
#pragma unroll
        for (int i = 0; i < K / 4; i++) {
            const float4 t = reinterpret_cast<const float4 *>(p)[i];
            v[4 * i] = t.x; v[4 * i + 1] = t.y; v[4 * i + 2] = t.z; v[4 * i + 3] = t.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < K; i++) v[i] = p[i];
    }
}

// Where chunk 0 of sample row b lands within its row (chunk c: at c ^ this).  Four consecutive rows differ
// in the chunk bits above a 32-channel group (transposed reads: 4 rows x 64 bytes at a time), sixteen rows in
// all chunk bits (row reads: the same chunk of 16 rows).
template <int CW> __device__ __forceinline__ int slab_swizzle(int b) {
    if constexpr (CW == 128) return ((b & 3) << 2) | ((b >> 2) & 3);
    else return ((b >> 3) & 1) | ((b >> 1) & 2) | ((b << 1) & 4);  // bits 1, 2, 3 of b, reversed (two rows per 256 bytes)
}

}  // namespace mhc
