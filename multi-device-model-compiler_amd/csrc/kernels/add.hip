// Elementwise fp32 add at the HBM roofline.
//
// Replaces the kernel the reference's pipeline generates for onnx.Add
// (1200 blocks x 1024 threads, one scalar element per thread:
// include/multi-device-model-compiler/Dialect/Device/Transform/Passes.td:86-89)
// with 128-bit loads and non-temporal 128-bit stores, one vector per lane and one
// block per 256 vectors (the grid is sized to the array, not to the machine: blocks
// are dispatched in index order, so the device sweeps one window of memory at a time).
// One IEEE add per element: bit exact with examples/add.ll:42-66.
#include "common.hpp"
#include "mgpu_ops_internal.hpp"

#include <algorithm>

namespace mgpu {

typedef float float4v __attribute__((ext_vector_type(4)));

// One vector per lane, one block per 256 vectors.  Measured on MI355X at the (3,640,640) shape: plain loads + non-temporal
// stores with one vector per lane is the fastest combination (non-temporal LOADS cost about 10 %, more vectors per lane do
// not help at this size).  The last n % 4 elements are one lane's, element by element: as a launch of their own they took
// as long as a small array (75850 elements 8.0 -> 4.1 us, 31136098 65 -> 63).
//
// Everything the kernel needs arrives as an explicit argument (the grid's stride included,
// instead of gridDim): the explicit arguments are preloaded into SGPRs, the grid dimensions
// would cost a load from the kernarg segment on the path to the first data load.
__global__ __launch_bounds__(256) void add_f32_vec4_kernel(const float *__restrict__ a, const float *__restrict__ b, float *__restrict__ c,
                                                           int64_t n, int64_t stride) {
  for (int64_t i = (int64_t)blockIdx.x * 1024 + threadIdx.x * 4; i < n; i += stride) {
    if (i + 4 <= n) {
      const float4v va = *reinterpret_cast<const float4v *>(a + i), vb = *reinterpret_cast<const float4v *>(b + i);
      __builtin_nontemporal_store(va + vb, reinterpret_cast<float4v *>(c + i));
    } else {
      for (int64_t j = i; j < n; j++) c[j] = a[j] + b[j];
    }
  }
}

// Pointers that are not 16-byte aligned.
__global__ __launch_bounds__(256) void add_f32_scalar_kernel(const float *__restrict__ a, const float *__restrict__ b, float *__restrict__ c,
                                                             int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) c[i] = a[i] + b[i];
}

void addF32(const float *a, const float *b, float *c, int64_t n, hipStream_t stream) {
  if (n < 0) fail("mgpuAddF32: negative element count");
  if (n == 0) return;
  if (!a || !b || !c) fail("mgpuAddF32: null pointer");
  if (aligned16(a) && aligned16(b) && aligned16(c)) {
    const int64_t blocks = std::min<int64_t>((n + 1023) / 1024, kMaxStreamBlocks);
    launchKernel(add_f32_vec4_kernel, dim3((unsigned)blocks), dim3(256), stream, a, b, c, n, blocks * 1024);
    MGPU_CHECK_LAUNCH("add_f32_vec4_kernel");
  } else {
    const int64_t blocks = std::min<int64_t>((n + 255) / 256, kMaxStreamBlocks);
    launchKernel(add_f32_scalar_kernel, dim3((unsigned)blocks), dim3(256), stream, a, b, c, n);
    MGPU_CHECK_LAUNCH("add_f32_scalar_kernel");
  }
}

} // namespace mgpu
