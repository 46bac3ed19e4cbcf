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

// Operands in pieces (conv_split.hip has the reasons): times the one scale each, their sums times the other.
constexpr int kPieces = 3;
constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-48f;

// a and b as three bf16 numbers each, the first of which is the nearest, the second the nearest to what that leaves: all 24 bits (as long
// as the last one is no subnormal: from 2^-110 on).  (v_cvt_pk_bf16_f32 by the compiler, not by inline assembly: a matrix instruction
// that reads its result needs two wait states behind it, which the compiler sees to only for instructions that it knows.)
__device__ __forceinline__ void splitTriple(float a, float b, uint32_t (&piece)[3]) {
#pragma unroll
  for (int i = 0; i < 3; i++) {
    piece[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
    a -= __builtin_bit_cast(float, piece[i] << 16);
    b -= __builtin_bit_cast(float, piece[i] & 0xffff0000u);
  }
}

} // namespace mgpu
