// tbq_dma.hpp -- direct global-to-LDS copies (gfx950 buffer_load_dwordx4 ...
// lds) for the MFMA kernels, with explicit waits.
//
// A copy moves 16 bytes per lane without passing through registers: lane i's
// 16 bytes at rsrc + voff(i) + soff land at LDS byte m0 + 16 i, so one
// wave's copy fills 1 KiB of LDS contiguously and the per-lane addresses
// choose what goes there (the XOR swizzles below are made this way).  The
// copy is written as asm because the compiler's wait-count pass waits for
// every outstanding copy before any LDS read it cannot prove unrelated; here
// the kernels wait themselves (dma_wait_barrier), once per step, for copies issued a
// whole step earlier.  The asm has no register output: nothing lands in a
// register the compiler could reuse early.
#pragma once

#include "tbq_device.hpp"

namespace tbq {

typedef int dma_rsrc_t __attribute__((ext_vector_type(4)));

// Buffer descriptor over [base, base + bytes): lanes past it read zeros.
__device__ __forceinline__ dma_rsrc_t dma_rsrc(const void *base, uint32_t bytes) {
    const uint64_t a = (uint64_t)base;
    dma_rsrc_t r;
    r.x = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
    r.y = __builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xFFFFu));
    r.z = __builtin_amdgcn_readfirstlane((int)bytes);
    r.w = 0x00020000;
    return r;
}

// LDS byte address of a pointer into __shared__ memory.
__device__ __forceinline__ uint32_t lds_addr(const void *p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)p;
}

// 1 KiB: lane i copies the 16 bytes at voff (per lane) + soff (uniform) to
// LDS byte lds + 16 i (lds uniform).
__device__ __forceinline__ void dma16(uint32_t lds, uint32_t voff, dma_rsrc_t rsrc, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(voff),
                 "s"(rsrc), "s"(soff)
                 : "memory");
}

// 256 bytes: lane i copies the 4 bytes at voff to LDS byte lds + 4 i.
__device__ __forceinline__ void dma4(uint32_t lds, uint32_t voff, dma_rsrc_t rsrc) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds" ::"s"(lds), "v"(voff), "s"(rsrc)
                 : "memory");
}

// dma16 from a 64-bit address per lane.
__device__ __forceinline__ void dma16_ptr(uint32_t lds, const void *p) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(p) : "memory");
}

// Every outstanding copy of this wave has landed and every LDS read it has
// issued has returned, then the workgroup's barrier: what the other waves
// copied is visible, and what this wave read may be overwritten.
__device__ __forceinline__ void dma_wait_barrier() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Every LDS read this wave has issued has returned: what it read may be
// overwritten by copies of its own (rows that no other wave reads).
__device__ __forceinline__ void lds_read_wait() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// dma_wait_barrier with the N memory operations issued last left in flight (they
// complete in issue order, so all copies before them have landed).
template <int N>
__device__ __forceinline__ void dma_wait_barrier_n() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

}  // namespace tbq
