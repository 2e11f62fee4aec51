// Products of 32 x 32 x 16 bf16 values by asm (latent attention's row tiles, prompts of head pairs).  Where a wave has its SIMD to itself what stands
// between the products is laid out by hand, and the compiler would sink an LDS read to its use (or hoist them all, into scratch): volatile with a
// memory clobber, each product stays between the reads around it.  The waits that the compiler then cannot see are the kernel's: two slots at the least between
// a VALU write of an operand and the product, MMA_WAIT between a last product and the first other reader of its result, without that
// result as an operand of the wait, as the compiler may copy an operand ahead of it.
#pragma once
#include "common.h"

#define MMA_WAIT "s_nop 15\n\ts_nop 3"
__device__ __forceinline__ void mma_add(f32x16& c, bf16x8 a, bf16x8 b) {   // c += a b, c in vector registers
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b) : "memory");
#endif
}
__device__ __forceinline__ void mma_acc(f32x16& c, bf16x8 a, bf16x8 b) {   // c += a b, c in accumulation registers
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b) : "memory");
#endif
}
