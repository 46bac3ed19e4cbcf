// What the convolution kernels share: division by numbers that the host knows, and buffer resources over fp32 tensors.
#pragma once

#include "common.hpp"
#include "mfma.hpp"

namespace mgpu {

constexpr int kOutside = (int)0x80000000; // a byte offset past every resource: the hardware's bounds check reads 0 there

// Division by a number that the host knows, for dividends below 2^31: (mulhi(n, mul) + n) >> shift.
struct FastDiv {
  unsigned mul, shift;
};
__device__ __forceinline__ int divide(int n, FastDiv d) {
  return (int)((__umulhi((unsigned)n, d.mul) + (unsigned)n) >> d.shift);
}
inline FastDiv fastDiv(int d) {
  unsigned shift = 0;
  while ((1u << shift) < (unsigned)d) shift++;
  return {(unsigned)((((uint64_t)1 << 32) * (((uint64_t)1 << shift) - d)) / d + 1), shift};
}

// A buffer resource over `elems` floats (2 GiB of them at most: no offset reaches further), for the
// builtins and, as its four words, for inline assembly.
constexpr int kRawBuffer = 0x00027000;
__device__ __forceinline__ int resourceBytes(int64_t elems) { return (int)(elems * 4 < 0x7fffffff ? elems * 4 : 0x7fffffff); }
__device__ __forceinline__ __amdgpu_buffer_rsrc_t resource(const float *p, int64_t elems) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), 0, resourceBytes(elems), kRawBuffer);
}
__device__ __forceinline__ i32x4 resourceWords(const float *p, int64_t elems) {
  const uint64_t at = (uint64_t)(uintptr_t)p;
  return i32x4{(int)(uint32_t)at, (int)(uint32_t)(at >> 32) & 0xffff, resourceBytes(elems), kRawBuffer};
}

// a and b as fp16 numbers, hi, and what these leave, lo: pairs of 22 bits where lo is no smaller than fp16's normal numbers, 2^-25
// off below.  (Four instructions; v_fma_mixlo / mixhi_f16 would be fewer where a scale comes besides, but writing half a register
// takes them two to three times as long.)
__device__ __forceinline__ void splitPair(float a, float b, uint32_t &hi, uint32_t &lo) {
  asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
  float ra, rb;
  asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[0,0,1]" : "=v"(ra) : "v"(a), "v"(hi));
  asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(rb) : "v"(b), "v"(hi));
  asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(lo) : "v"(ra), "v"(rb));
}

// a and b as three bf16 numbers each, the first of which is the nearest, the second the nearest to what that leaves: all 24 bits (as long
// as the last one is no subnormal: from 2^-110 on).
__device__ __forceinline__ void splitTriple(float a, float b, uint32_t (&piece)[3]) {
#pragma unroll
  for (int i = 0; i < 3; i++) {
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(piece[i]) : "v"(a), "v"(b));
    a -= __builtin_bit_cast(float, piece[i] << 16);
    b -= __builtin_bit_cast(float, piece[i] & 0xffff0000u);
  }
}

} // namespace mgpu
