// A layer's weights from fp32 to fp16 in one launch: the arrays' table and what one block does, for the kernel that casts them
// alone (cast.hip) and the one that also casts and normalises the layer's input (layernorm.hip).
#pragma once

#include "common.hpp"
#include "mfma.hpp"
#include "mgpu_ops_internal.hpp"
#include "types.hpp"

namespace mgpu {

// The reference layer hands over fp32 weights on every call; casting its seven arrays one by one is seven
// launches of 2.3 us host time, most of them a few microseconds of work.  Here one grid covers them all: a block finds
// its array among the first-block numbers in the arguments.  A plain array goes 8 elements a lane and vector, four vectors ahead of
// the first store (bound by memory: beside a LayerNorm, whose registers leave a CU five wavefronts a SIMD, one vector a lane would
// be too few loads in flight: decoding layer of 2048, ffn 8192, on 84 tokens 116 us, four 107, the two kernels in turn 109); one wanted
// K-major (transposed) goes in 64 x 64 tiles, four rows by four columns per thread, through LDS at a pitch of
// 68 halves: 16 bytes a lane from and to memory, 8-byte LDS accesses that meet every bank equally often
// (d_model 2048, ffn 2048, 151 MB: 26 us, 5.8 TB/s).
struct CastTable {
  CastJob job[kMaxCastJobs];
  unsigned firstBlock[kMaxCastJobs + 1];
  int count;
};
constexpr int kPlainVectors = 4; // of 8 elements a lane
constexpr int kPlainPerBlock = 2048 * kPlainVectors;

// A thread block's share: number `at` of the table's (256 threads, whole in the call).
__device__ __forceinline__ void castTableBlock(const CastTable &t, unsigned at) {
  __shared__ __attribute__((aligned(16))) _Float16 tile[64][68];
  int j = 0;
  while (j + 1 < t.count && at >= t.firstBlock[j + 1]) j++; // (uniform)
  const CastJob job = t.job[j];
  const unsigned block = at - t.firstBlock[j];
  const float *src = job.src;
  _Float16 *dst = static_cast<_Float16 *>(job.dst);
  const int tid = threadIdx.x;
  if (!job.kMajor) {
    const int64_t n = job.rows * job.cols, first = (int64_t)block * kPlainPerBlock + tid * 8;
    if (job.vector && (int64_t)(block + 1) * kPlainPerBlock <= n) { // (uniform: every load ahead of the first store)
      f32x4 v[kPlainVectors][2];
#pragma unroll
      for (int k = 0; k < kPlainVectors; k++) {
        v[k][0] = *reinterpret_cast<const f32x4 *>(src + first + k * 2048);
        v[k][1] = *reinterpret_cast<const f32x4 *>(src + first + k * 2048 + 4);
      }
#pragma unroll
      for (int k = 0; k < kPlainVectors; k++) {
        const float x[8] = {v[k][0][0], v[k][0][1], v[k][0][2], v[k][0][3], v[k][1][0], v[k][1][1], v[k][1][2], v[k][1][3]};
        *reinterpret_cast<u32x4 *>(dst + first + k * 2048) = ElemTraits<_Float16>::pack(x);
      }
      return;
    }
    for (int64_t i = first; i < first + kPlainPerBlock && i < n; i += 2048) {
      if (job.vector && i + 8 <= n) {
        const f32x4 lo = *reinterpret_cast<const f32x4 *>(src + i), hi = *reinterpret_cast<const f32x4 *>(src + i + 4);
        const float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        *reinterpret_cast<u32x4 *>(dst + i) = ElemTraits<_Float16>::pack(x);
      } else {
        for (int e = 0; e < 8; e++)
          if (i + e < n) dst[i + e] = (_Float16)src[i + e];
      }
    }
    return;
  }
  const int64_t tilesC = (job.cols + 63) / 64;
  const int64_t r0 = (int64_t)(block / tilesC) * 64, c0 = (int64_t)(block % tilesC) * 64;
  const bool whole = job.vector && r0 + 64 <= job.rows && c0 + 64 <= job.cols; // (uniform)
  const int q = tid % 16, w = tid / 16; // this thread: rows 4 w.., columns 4 q..
  f32x4 v[4];
  if (whole) {
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = *reinterpret_cast<const f32x4 *>(src + (r0 + 4 * w + i) * job.cols + c0 + 4 * q);
  } else {
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int64_t r = r0 + 4 * w + i, c = c0 + 4 * q + e;
        v[i][e] = r < job.rows && c < job.cols ? src[r * job.cols + c] : 0.0f;
      }
  }
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const f16x4 col = {(_Float16)v[0][e], (_Float16)v[1][e], (_Float16)v[2][e], (_Float16)v[3][e]};
    *reinterpret_cast<f16x4 *>(&tile[4 * q + e][4 * w]) = col;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int c = tid / 8 + 32 * i, r = 8 * (tid % 8);
    const f16x4 lo = *reinterpret_cast<const f16x4 *>(&tile[c][r]), hi = *reinterpret_cast<const f16x4 *>(&tile[c][r + 4]);
    _Float16 *out = dst + (c0 + c) * job.rows + r0 + r;
    if (whole) {
      *reinterpret_cast<f16x8 *>(out) = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    } else if (c0 + c < job.cols) {
#pragma unroll
      for (int e = 0; e < 8; e++)
        if (r0 + r + e < job.rows) out[e] = e < 4 ? lo[e % 4] : hi[e % 4];
    }
  }
}

// The table of these arrays (their `vector` is set here), and the blocks of 256 threads that it takes.
unsigned castTable(CastJob *jobs, int count, CastTable &t);

} // namespace mgpu
