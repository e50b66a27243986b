// Loads straight from global memory into LDS, and the waits and barriers that go with them.  Such a load is issued from an
// asm statement, so the compiler keeps no book on it: it neither waits for these loads before LDS reads it cannot tell
// apart from their destination, nor turns its other waits into waits for everything.  The caller counts them (wait_vmcnt) and
// orders LDS accesses around them (barrier_no_drain).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bitsmoe {

// LDS element offset of the 16-byte chunk c (0..7) of row r of a stage of rows of 64 16-bit values: rows are 128
// bytes apart without padding, and the chunks of a row are permuted by the row index so that the
// sixteen rows an MFMA operand load touches fall into different banks.  (LDS-direct loads fill
// LDS in lane order, which rules out padded rows.)
__device__ __forceinline__ int dma_chunk_off(int r, int c) { return r * 64 + ((c ^ ((r >> 1) & 7)) << 3); }

// s_waitcnt that only waits for the vector-memory counter: at most `n` operations outstanding
// (the counter is six bits wide, split over the immediate; the other counters are left alone).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "the counter is six bits wide");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | 0x0F70);
}
// s_waitcnt lgkmcnt(0) alone: every LDS read of the wavefront has returned (the vector-memory and
// export counters are left at their maxima).
__device__ __forceinline__ void wait_lds_reads() { __builtin_amdgcn_s_waitcnt(0xC07F); }
// Workgroup barrier without the wait for outstanding loads that __syncthreads implies.  The empty
// asm statements keep the compiler from moving LDS accesses across it (the bare instruction is no
// memory fence for the compiler).
__device__ __forceinline__ void barrier_no_drain() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// LDS-direct load: every active lane fetches 16 bytes from `src`, and the wavefront's data lands in
// LDS at lds_base + 16 * lane (lds_base is wave-uniform).
__device__ __forceinline__ void load_to_lds16(const void* src, void* lds_base) {
    using lvoid = void __attribute__((address_space(3)))*;
    const uint32_t l = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lvoid)lds_base);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(l) : "m0", "memory");
}
// The same from a wave-uniform base and 32 bits of byte offset per lane, to an LDS address (lds_address): no 64-bit address
// arithmetic per lane and load.
__device__ __forceinline__ void load_to_lds16(const void* base, uint32_t offset, uint32_t lds_at) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(offset), "s"(base), "s"(lds_at) : "m0", "memory");
}
__device__ __forceinline__ uint32_t lds_address(void* lds) {
    using lvoid = void __attribute__((address_space(3)))*;
    return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lvoid)lds);
}

}  // namespace bitsmoe
