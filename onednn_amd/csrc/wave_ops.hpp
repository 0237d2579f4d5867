// What the tile kernels' loops and epilogues share: direct-to-LDS loads, LDS reads by 32-bit address, scalar pinning,
// hand-counted waits.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace mi355 {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

namespace gemm {

// 4 bytes per lane: LDS byte address lds_addr + 4*i
__device__ __forceinline__ void dma4(const void *sbase, unsigned voff, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(sbase)
                 : "memory", "m0");
}

// one wavefront-wide direct-to-LDS load: lane i brings 16 bytes from
// sbase + voff to LDS byte address lds_addr + 16*i
__device__ __forceinline__ void dma16(const void *sbase, unsigned voff, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(sbase)
                 : "memory", "m0");
}

// LDS reads through explicit 32-bit LDS addresses: a generic pointer that the
// compiler cannot prove to be shared memory (one selected between two stages,
// say) turns every ds_read into a flat load through the vector memory path.
typedef const v4i __attribute__((address_space(3))) *lds_v4i_ptr_t;
typedef const unsigned __attribute__((address_space(3))) *lds_u32_ptr_t;
__device__ __forceinline__ v4i lds_read16(unsigned addr) { return *(lds_v4i_ptr_t)(size_t)addr; }
__device__ __forceinline__ unsigned lds_read4(unsigned addr) { return *(lds_u32_ptr_t)(size_t)addr; }

// A workgroup-uniform value pinned to scalar registers: the DMA's base operand
// must be an SGPR pair, and a uniform value that merges at the join of divergent
// code ahead of the K loop counts as divergent from there on.  The value passes
// through an empty asm statement as a vector register, which hides from the
// compiler that it is uniform (it would fold a readfirstlane of a known-uniform
// value away, wherever it keeps it); the readfirstlane itself is the builtin, so
// that the compiler places the wait states the instruction needs after a VALU
// write of its source and before a memory instruction reads its result (an
// inline-assembly v_readfirstlane gets none of them: it read a stale register
// right behind the v_mov that fed it).
__device__ __forceinline__ int scalar_int(int x) {
    asm volatile("" : "+v"(x));
    int r = __builtin_amdgcn_readfirstlane(x);
    // the result may go straight into the base operand of a DMA written in inline
    // assembly, whose wait states after a VALU write of an SGPR (five before a
    // memory instruction reads it) the compiler cannot place either
    asm volatile("s_nop 4" : "+s"(r));
    return r;
}
__device__ __forceinline__ const char *scalar_ptr(const char *p) {
    const uint64_t v = (uint64_t)(uintptr_t)p;
    const uint32_t lo = (uint32_t)scalar_int((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)scalar_int((int)(uint32_t)(v >> 32));
    return (const char *)(uintptr_t)(((uint64_t)hi << 32) | lo);
}

// s_waitcnt vmcnt(n) only (expcnt / lgkmcnt left at their maxima)
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 0xF) | ((N >> 4) << 14));
}

// s_waitcnt lgkmcnt(0) only
__device__ __forceinline__ void wait_lds_reads() {
    __builtin_amdgcn_s_waitcnt(0xC07F);
}

// workgroup barrier that neither memory accesses nor MFMAs are scheduled across
__device__ __forceinline__ void phase_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
}

} // namespace gemm
} // namespace mi355
