// What follows a GEMM whose reduction was split over blocks (gemmPartial*): the fp32 planes of partial sums are added up,
// with the bias and the residual, by the kernel that reads the product next anyway - the residual add + LayerNorm between
// two blocks of a layer, or the conversion of a layer's result to fp32.
//
// A wavefront owns a row and keeps it in registers (8 columns per lane and vector, N <= 2048), every load of the row in
// flight at once: one trip to memory, two passes over the registers for the statistics.  That trip bounds it at the few
// rows this is used for: (77, 768), three planes 3.2 us (5.1 with the planes loaded one after another) against 3.0
// for the LayerNorm of one fp16 product; (1368, 768) 4.7 against 4.0.
#include "common.hpp"
#include "mgpu_ops_internal.hpp"
#include "types.hpp"

namespace mgpu {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float waveSum(float v) {
#pragma unroll
  for (int d = 32; d > 0; d /= 2) v += __shfl_xor(v, d);
  return v;
}

// Sum: the fp32 sum to out.  Norm: LayerNorm(sum) in fp16, and the rounded sum to sumOut when it is not null.  NormF32: in fp32.
enum class Result { Sum, Norm, NormF32 };
template <int V, int PARTS, Result RESULT>
__global__ __launch_bounds__(64) void partial_sums_kernel(const float *__restrict__ planes, const _Float16 *__restrict__ bias,
                                                          const _Float16 *__restrict__ residual, const _Float16 *__restrict__ gamma,
                                                          const _Float16 *__restrict__ beta, _Float16 *__restrict__ sumOut,
                                                          void *__restrict__ out, int M, int N, float eps) {
  constexpr bool NORM = RESULT != Result::Sum;
  const int row = blockIdx.x, lane = threadIdx.x;
  // every load first, so that one trip to memory covers them all (columns past the row fetch its last vector)
  float4v p[V][PARTS][2];
  half8 b[V], r[V], g[V], be[V];
#pragma unroll
  for (int v = 0; v < V; v++) {
    const int n = (v * 64 + lane) * 8 < N ? (v * 64 + lane) * 8 : N - 8;
    const float *from = planes + (size_t)row * N + n;
#pragma unroll
    for (int q = 0; q < PARTS; q++) {
      p[v][q][0] = *reinterpret_cast<const float4v *>(from + (size_t)q * M * N);
      p[v][q][1] = *reinterpret_cast<const float4v *>(from + (size_t)q * M * N + 4);
    }
    b[v] = *reinterpret_cast<const half8 *>(bias + n);
    r[v] = *reinterpret_cast<const half8 *>(residual + (size_t)row * N + n);
    if (NORM) {
      g[v] = *reinterpret_cast<const half8 *>(gamma + n);
      be[v] = *reinterpret_cast<const half8 *>(beta + n);
    }
  }
  float x[V][8];
  float sum = 0.0f;
#pragma unroll
  for (int v = 0; v < V; v++) {
    const int n = (v * 64 + lane) * 8;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      x[v][i] = 0.0f;
#pragma unroll
      for (int q = 0; q < PARTS; q++) x[v][i] += p[v][q][i / 4][i % 4];
      x[v][i] += (float)b[v][i];
      x[v][i] += (float)r[v][i];
    }
    if (n >= N) continue;
#pragma unroll
    for (int i = 0; i < 8; i++) sum += x[v][i];
    if (!NORM) {
      float *o = static_cast<float *>(out) + (size_t)row * N + n;
      *reinterpret_cast<float4v *>(o) = float4v{x[v][0], x[v][1], x[v][2], x[v][3]};
      *reinterpret_cast<float4v *>(o + 4) = float4v{x[v][4], x[v][5], x[v][6], x[v][7]};
    } else if (sumOut) {
      half8 s;
#pragma unroll
      for (int i = 0; i < 8; i++) s[i] = (_Float16)x[v][i];
      *reinterpret_cast<half8 *>(sumOut + (size_t)row * N + n) = s;
    }
  }
  if (!NORM) return;
  const float mean = waveSum(sum) / (float)N;
  float sq = 0.0f;
#pragma unroll
  for (int v = 0; v < V; v++)
    if ((v * 64 + lane) * 8 < N)
#pragma unroll
      for (int i = 0; i < 8; i++) sq += (x[v][i] - mean) * (x[v][i] - mean);
  const float inv = 1.0f / sqrtf(waveSum(sq) / (float)N + eps);
#pragma unroll
  for (int v = 0; v < V; v++) {
    const int n = (v * 64 + lane) * 8;
    if (n >= N) continue;
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; i++) y[i] = (x[v][i] - mean) * inv * (float)g[v][i] + (float)be[v][i];
    if (RESULT == Result::NormF32) {
      float *o = static_cast<float *>(out) + (size_t)row * N + n;
      *reinterpret_cast<float4v *>(o) = float4v{y[0], y[1], y[2], y[3]};
      *reinterpret_cast<float4v *>(o + 4) = float4v{y[4], y[5], y[6], y[7]};
      continue;
    }
    half8 o;
#pragma unroll
    for (int i = 0; i < 8; i++) o[i] = (_Float16)y[i];
    *reinterpret_cast<half8 *>(static_cast<_Float16 *>(out) + (size_t)row * N + n) = o;
  }
}

template <int PARTS, Result RESULT>
void launch(const float *planes, const void *bias, const void *residual, const void *gamma, const void *beta, void *sumOut, void *out,
            float eps, int64_t M, int64_t N, hipStream_t stream) {
  const dim3 grid((unsigned)M), block(64);
  const auto *b = static_cast<const _Float16 *>(bias), *r = static_cast<const _Float16 *>(residual);
  const auto *g = static_cast<const _Float16 *>(gamma), *be = static_cast<const _Float16 *>(beta);
  auto *s = static_cast<_Float16 *>(sumOut);
  const auto kernel = N <= 512 ? partial_sums_kernel<1, PARTS, RESULT> : N <= 1024 ? partial_sums_kernel<2, PARTS, RESULT>
                                                                                   : partial_sums_kernel<4, PARTS, RESULT>;
  launchKernel(kernel, grid, block, stream, planes, b, r, g, be, s, out, (int)M, (int)N, eps);
  MGPU_CHECK_LAUNCH("partial_sums_kernel");
}

template <Result RESULT, typename... Args> void launchParts(int parts, Args... args) {
  if (parts == 2) launch<2, RESULT>(args...);
  else if (parts == 3) launch<3, RESULT>(args...);
  else if (parts == 4) launch<4, RESULT>(args...);
  else fail("partialSums: internal dispatch error");
}

} // namespace

bool partialSumsSupports(const void *bias, const void *residual, const void *gamma, const void *beta, const void *out, int64_t M, int64_t N) {
  return M <= 0x7fffffff && N > 0 && N % 8 == 0 && N <= 2048 && aligned16(bias) && aligned16(residual) && aligned16(gamma) && aligned16(beta) && aligned16(out);
}

void partialSumsLayerNormF16(const float *planes, int parts, const void *bias, const void *residual, const void *gamma, const void *beta,
                             void *sumOut, void *out, float eps, int64_t M, int64_t N, hipStream_t stream) {
  launchParts<Result::Norm>(parts, planes, bias, residual, gamma, beta, sumOut, out, eps, M, N, stream);
}

void partialSumsLayerNormF32(const float *planes, int parts, const void *bias, const void *residual, const void *gamma, const void *beta,
                             float *out, float eps, int64_t M, int64_t N, hipStream_t stream) {
  launchParts<Result::NormF32>(parts, planes, bias, residual, gamma, beta, nullptr, out, eps, M, N, stream);
}

void partialSumsF32(const float *planes, int parts, const void *bias, const void *residual, float *out, int64_t M, int64_t N,
                    hipStream_t stream) {
  launchParts<Result::Sum>(parts, planes, bias, residual, nullptr, nullptr, nullptr, out, 0.0f, M, N, stream);
}

} // namespace mgpu
