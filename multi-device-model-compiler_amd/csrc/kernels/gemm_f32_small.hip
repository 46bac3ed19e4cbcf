// fp32 GEMM for few tiles: out[M,N] = act(in[M,K] . W[K,N] + bias[N]) (+ residual[M,N]), any M, N, K.
//
// True fp32 products on the matrix cores (v_mfma_f32_32x32x2_f32).  A block owns a 32 x 32 tile and its
// eight wavefronts split the reduction; operands go straight from L1 / L2 to registers - lane half hl takes
// k 4 hl .. 4 hl + 3 of an 8-k chunk, the input by a 16-byte load along a row, the weight by rows of 32
// columns - a chunk ahead of the MFMAs.  The partial tiles meet in LDS.  Rows and columns past the end are
// read from the last ones and not stored; k past the end is zero on both sides.
// Bound by launch and one round trip to memory: 96 x 64 x 32 2.5 us (library 4.5), 512 x 512 x 512 6.1 (6.7);
// beyond (gemm.cpp has the line) an operand byte is re-read too often from L2 and the library is ahead.
#include "common.hpp"
#include "mgpu_ops_internal.hpp"

namespace mgpu {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8;
constexpr int kHalf = 4, kChunk = 2 * kHalf; // k of a step, kHalf per lane half (4: 6.1 us at 512^3, 8: 6.7, 16: 6.8)

template <int ACT>
__global__ __launch_bounds__(64 * kWaves, 2) void gemm_f32_small_kernel(const float *__restrict__ in, const float *__restrict__ weight,
                                                                        const float *__restrict__ bias, const float *residual, float *out,
                                                                        int M, int N, int K, int tilesM) {
  __shared__ float partial[kWaves][16 * 64];
  const int tid = threadIdx.x, lane = tid % 64;
  const int ks = __builtin_amdgcn_readfirstlane(tid / 64);
  const int l32 = lane % 32, hl = lane / 32;
  const int m0 = (int)(blockIdx.x % tilesM) * 32, n0 = (int)(blockIdx.x / tilesM) * 32;
  const float *xrow = in + (int64_t)(m0 + l32 < M ? m0 + l32 : M - 1) * K;
  const float *wcol = weight + (n0 + l32 < N ? n0 + l32 : N - 1);

  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; i++) acc[i] = 0.0f;
  struct Operands {
    float a[kHalf], b[kHalf];
  };
  auto fetch = [&](Operands &o, int k0) {
    const int k = k0 + kHalf * hl;
    if (k0 + kChunk <= K) { // (uniform)
#pragma unroll
      for (int i = 0; i < kHalf; i += 4) {
        const f32x4 v = *reinterpret_cast<const f32x4 __attribute__((aligned(4))) *>(xrow + k + i);
#pragma unroll
        for (int e = 0; e < 4; e++) o.a[i + e] = v[e];
      }
#pragma unroll
      for (int i = 0; i < kHalf; i++) o.b[i] = wcol[(int64_t)(k + i) * N];
    } else {
#pragma unroll
      for (int i = 0; i < kHalf; i++) {
        const bool in = k + i < K;
        const float a = xrow[in ? k + i : 0], b = wcol[in ? (int64_t)(k + i) * N : 0];
        o.a[i] = in ? a : 0.0f;
        o.b[i] = in ? b : 0.0f;
      }
    }
  };
  auto multiply = [&](const Operands &o) {
#pragma unroll
    for (int i = 0; i < kHalf; i++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(o.a[i], o.b[i], acc, 0, 0, 0);
  };
  const int chunks = (K + kChunk - 1) / kChunk;
  const int c0 = chunks * ks / kWaves, c1 = chunks * (ks + 1) / kWaves;
  Operands even, odd;
  if (c0 < c1) fetch(even, c0 * kChunk);
  for (int c = c0; c < c1; c += 2) {
    if (c + 1 < c1) fetch(odd, (c + 1) * kChunk);
    multiply(even);
    if (c + 1 >= c1) break;
    if (c + 2 < c1) fetch(even, (c + 2) * kChunk);
    multiply(odd);
  }

  // accumulator register r of lane l: row 8*(r/4) + 4*(l/32) + r%4, column l%32; two registers per wavefront
#pragma unroll
  for (int r = 0; r < 16; r++) partial[ks][r * 64 + lane] = acc[r];
  __syncthreads();
  const int n = n0 + l32;
  const float bv = bias && n < N ? bias[n] : 0.0f;
#pragma unroll
  for (int i = 0; i < 16 / kWaves; i++) {
    const int r = ks * (16 / kWaves) + i;
    const int m = m0 + 8 * (r / 4) + 4 * hl + r % 4;
    float v = 0.0f;
#pragma unroll
    for (int s = 0; s < kWaves; s++) v += partial[s][r * 64 + lane];
    if (m >= M || n >= N) continue;
    v += bv;
    if (ACT == ACT_RELU) v = v > 0.0f ? v : 0.0f;
    if (ACT == ACT_GELU) v = gelu_erf(v);
    if (residual) v += residual[(int64_t)m * N + n];
    out[(int64_t)m * N + n] = v;
  }
}

} // namespace

void gemmF32Small(const float *in, const float *weight, const float *bias, const float *residual, float *out, int64_t M, int64_t N, int64_t K,
                  int act, hipStream_t stream) {
  const int tilesM = (int)((M + 31) / 32), tilesN = (int)((N + 31) / 32);
  const dim3 grid((unsigned)(tilesM * tilesN)), block(64 * kWaves);
  if (act == ACT_RELU)
    launchKernel(gemm_f32_small_kernel<ACT_RELU>, grid, block, stream, in, weight, bias, residual, out, (int)M, (int)N, (int)K, tilesM);
  else if (act == ACT_GELU)
    launchKernel(gemm_f32_small_kernel<ACT_GELU>, grid, block, stream, in, weight, bias, residual, out, (int)M, (int)N, (int)K, tilesM);
  else
    launchKernel(gemm_f32_small_kernel<ACT_NONE>, grid, block, stream, in, weight, bias, residual, out, (int)M, (int)N, (int)K, tilesM);
  MGPU_CHECK_LAUNCH("gemm_f32_small_kernel");
}

} // namespace mgpu
