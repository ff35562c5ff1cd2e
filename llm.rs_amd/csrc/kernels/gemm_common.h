// gemm_common.h - what the tile GEMM (prefill.hip) and the skinny GEMM
// (sgemm.hip) share: loads straight to LDS, an ordering aid, and the plain
// block loop of one output.
#pragma once
#include "common.h"
#include "gemv_core.h"
#include "../kernel_args.h"

namespace llmrs {

// The value is computed here and read after here.
template <typename T>
__device__ __forceinline__ void pin(T& x) {
  asm volatile("" : "+v"(x));
}

// 16 (4) bytes per lane from global memory to lds + 16 (4) * lane, without
// registers.
__device__ __forceinline__ void load_lds16(const void* src, uint8_t* lds) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                   (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}
__device__ __forceinline__ void load_lds4(const void* src, uint8_t* lds) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                   (__attribute__((address_space(3))) void*)lds, 4, 0, 0);
}

template <int WT>
__device__ __forceinline__ unsigned load_scale(const void* ws, size_t i) {
  return WT == WT_Q4F ? ((const unsigned*)ws)[i] : ((const uint16_t*)ws)[i];
}

// q - 8 for four nibbles held one per byte (0..15): (v + 0x78) ^ 0x80 per
// byte, no carry between bytes.
__device__ __forceinline__ unsigned nib_s8(unsigned v) { return (v + 0x78787878u) ^ 0x80808080u; }

// Codes carried as 16 (q - 8) make every term and partial sum 16 times the
// reference's: the same bits with another exponent (products and sums below
// the normal range are exact on both sides), until one passes 2^124 and
// overflows where the reference's is finite.  An overflow stays in the total
// as an infinity or NaN, so a finite total had none.
__device__ __forceinline__ bool is_finite(float x) { return __builtin_fabsf(x) < INFINITY; }

// Output (token t, row n) by the reference's own loop (cpu.rs:910-937), for
// the totals that are not finite: unscaled codes, one block after the other.
// Rare, so it is kept small: any Args with xq, xd, wq, ws and K.
template <int WT, int LAYOUT, typename Args>
__device__ float q4_block_loop(const Args& a, int t, int n) {
  static_assert(WT != WT_Q8H, "Q8 codes are not scaled");
  const int nb = a.K >> 5;
  const int8_t* x = a.xq + act_row(t, a.K, LAYOUT);
  const float* xd = a.xd + act_scale_row(t, nb, LAYOUT);
  float total = 0.0f;
  // a NaN stays one; rows with infinite scales come to it within a few blocks, so
  // that a launch full of them is not left to this loop
#pragma unroll 1
  for (int b = 0; b < nb && total == total; ++b) {
    const size_t wb = (size_t)n * nb + b;
    int isum = 0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {  // dword g: elements 4 g .. in the low nibbles, 16 + 4 g .. in the high
      const unsigned w = ((const unsigned*)(a.wq + wb * 16))[g];
      const int lo = *(const int*)(x + act_offset(32 * b + 4 * g, LAYOUT));
      const int hi = *(const int*)(x + act_offset(32 * b + 16 + 4 * g, LAYOUT));
      isum = dot4((int)nib_s8(w & 0x0F0F0F0Fu), lo, isum);
      isum = dot4((int)nib_s8((w >> 4) & 0x0F0F0F0Fu), hi, isum);
    }
    total = total + (float)isum * (wscale<WT>(load_scale<WT>(a.ws, wb)) * xd[act_scale_offset(b, LAYOUT)]);
  }
  return total;
}

}  // namespace llmrs
