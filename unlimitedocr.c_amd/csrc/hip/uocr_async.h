/*
 * uocr_async.h - loads straight into LDS, counted by the wavefront itself.
 */
#ifndef UOCR_ASYNC_H
#define UOCR_ASYNC_H

#include "uocr_gemm.h"

/* Waits until at most N of the wavefront's vector memory operations are in
 * flight and its LDS reads are done, then for the block's other wavefronts. */
template <int N>
__device__ __forceinline__ void wait_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

__device__ __forceinline__ u32 uni(u32 v) {
    return (u32)__builtin_amdgcn_readfirstlane((int)v);
}

template <typename T>
__device__ __forceinline__ T *uni(T *p) {
    const uint64_t v = (uint64_t)p;
    return (T *)(((uint64_t)uni((u32)(v >> 32)) << 32) | uni((u32)v));
}

/* 16 bytes per lane from base + voff straight into LDS at lds + 16 lane.  In
 * inline assembly because the compiler's own LDS-direct load makes every later
 * LDS read wait for all of them; wait_barrier counts them instead.  m0 holds
 * the LDS address and is named as changed; the compiler warns that it reserves
 * the register, yet only so it does not keep a value of its own there across
 * the statement. */
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_load16(const void *base, u32 voff, u32 lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(voff), "s"(uni(base)), "s"(lds)
                 : "memory", "m0");
}
#pragma clang diagnostic pop

#endif /* UOCR_ASYNC_H */
