// Launcher of the fused multi-head attention kernel (fmha_kernel.hpp): picks the tile
// geometry and the instantiation for a head size and a mask, checks the operands.  Launches that would leave most of
// the chip idle go to fmha_split.hip.
//
// Replaces the dispatcher of the reference's cubin kernels, FusedMHARunnerFP16v2
// (3rdparty/trt_fused_multihead_attention/qkvToContext.cu:162-199,306-315;
// fused_multihead_attention_v2.h:5278-5377), called at lib/Kernels/GPU/LLM.cu:79-81.
#include "fmha_kernel.hpp"
#include "mgpu_ops_internal.hpp"

namespace mgpu {

namespace {

using namespace fmha_detail;

// Compute units of the current device (asked once per device).
int deviceComputeUnits() {
  static int cached[64]; // 0 = not asked yet
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int v = __atomic_load_n(&cached[dev], __ATOMIC_RELAXED);
  if (v == 0) {
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
    __atomic_store_n(&cached[dev], v, __ATOMIC_RELAXED);
  }
  return v;
}

// dHead: head dimension in memory; D: the tile geometry it runs in (dHead == D, or a
// smaller multiple of 8, up to USED, with the PAD instantiation).
template <typename T, int D, int NQ, bool PAD, int USED = D>
void launch(const void *qkv, const int32_t *seqlens, const int32_t *cuSeqlens, void *out, int B, int S, int H,
            int dHead, float scale, bool causal, hipStream_t stream) {
  constexpr int BM = 128 * NQ;
  const int nQB = (S + BM - 1) / BM;
  // Causal query blocks go in pairs of equal total work - block i with block nQB - 1 - i in one work
  // item - when there are exactly four of them (449 <= S <= 512), the head dimension is 64 or 128 (at
  // 256 the loop over the pair does not fit the registers of two wavefronts per SIMD) and the halved
  // grid still gives every CU two blocks.  Everywhere else handing the blocks out longest first (below)
  // measured as fast or faster than pairing: b16 s768 h12 d128 49.9 against 60.8 us, b2 s4096 h16 d64 84.8
  // against 92.3, b16 s640 h16 d64 28.8 against 30.6; at four blocks pairing wins by 4-12 %.
  const bool pair = causal && D <= 128 && nQB == 4 && (int64_t)B * H * 2 >= 2 * (int64_t)deviceComputeUnits();
  const int64_t blocks = (int64_t)B * H * (pair ? (nQB + 1) / 2 : nQB);
  // what the kernel is told: 1 = paired; 2 = unpaired causal blocks longest first (once compute units
  // hold more than one block); 0 = query blocks in index order
  const int order = pair ? 1 : (causal && blocks > deviceComputeUnits()) ? 2 : 0;
  if (blocks > 0x7fffffffLL) fail("fusedMHA: problem too large for one launch");
  const float c = scale * 1.44269504088896340736f;
  const auto *in = static_cast<const uint16_t *>(qkv);
  auto *o = static_cast<uint16_t *>(out);
  const dim3 grid((unsigned)blocks), block(256);
  // Two sets of wavefronts a block where a launch leaves every CU about one block, one wavefront a SIMD, and each set still has a
  // few tiles (us, one set / two, b x s x heads): 256 blocks 2 x 1024 x 16 of 64 16.9 / 14.5, 1 x 2048 x 16 of 128 46.0 / 41.4, of 256 103 / 91,
  // 192 1 x 3072 x 8 of 128 61.9 / 49.5, 4 x 512 x 16 of 64 10.1 / 9.5; but 7 x 384 x 12 of 128 13.9 / 15.3, 3 x 600 x 12 of 256 37.1 / 38.1, and
  // 264 blocks, a second round, 1 x 2697 x 12 of 128 74 / 93.  Causal launches end with a few long blocks: 352 2 x 1374 x 16 of 64 24.8 /
  // 19.8, 384 1 x 3000 x 16 of 128 67 / 56, 3 x 1024 x 16 19.7 / 18.5, 512 1 x 4096 x 16 100 / 86, but 360 6 x 640 x 12 14.0 / 15.9, 448 4 x 1024 x 14
  // 19.9 / 20.8, 640 1 x 4096 x 20 72 / 77.
  if constexpr (NQ == 1) {
    const int64_t cus = deviceComputeUnits();
    const bool halves = causal ? S >= 512 && !pair && 2 * blocks <= cus * (nQB >= 12 ? 4 : nQB >= 8 ? 3 : 2)
                               : S >= (D == 256 ? 768 : 512) && blocks <= cus;
    if (halves) {
      auto *kernel = causal ? fmha_fwd_kernel<T, D, 1, true, false, PAD, true, false, USED> : fmha_fwd_kernel<T, D, 1, false, false, PAD, true, false, USED>;
      launchKernel(kernel, grid, dim3(512), stream, in, seqlens, cuSeqlens, o, S, H, nQB, c, order, (int)blocks, dHead, nullptr);
      MGPU_CHECK_LAUNCH("fmha_fwd_kernel");
      return;
    }
  }
  if (causal) {
    // (the causal kernel exists with one 32-query block per wavefront only)
    if constexpr (NQ == 1)
      launchKernel(fmha_fwd_kernel<T, D, NQ, true, false, PAD, false, false, USED>, grid, block, stream, in, seqlens, cuSeqlens, o, S, H, nQB, c, order, (int)blocks, dHead, nullptr);
    else
      fail("fusedMHA: internal dispatch error");
  } else if (D == 128 && S <= 64 && (PAD || blocks <= deviceComputeUnits())) { // one tile of keys (the kernel has the times)
    launchKernel(fmha_fwd_kernel<T, D, NQ, false, false, PAD, false, D == 128, USED>, grid, block, stream, in, seqlens, cuSeqlens, o, S, H, nQB, c, order, (int)blocks, dHead, nullptr);
  } else {
    launchKernel(fmha_fwd_kernel<T, D, NQ, false, false, PAD, false, false, USED>, grid, block, stream, in, seqlens, cuSeqlens, o, S, H, nQB, c, order, (int)blocks, dHead, nullptr);
  }
  MGPU_CHECK_LAUNCH("fmha_fwd_kernel");
}

template <typename T>
void launchForHeadDim(const void *qkv, const int32_t *seqlens, const int32_t *cuSeqlens, void *out, int B, int S, int H,
                      int dHead, float scale, bool causal, hipStream_t stream) {
  // One 32-query block per wavefront, except on long unmasked-or-padded sequences at
  // head_dim 64: with 64 queries per wavefront every K / V operand read from LDS feeds
  // two MFMAs and a block of 256 queries shares each tile load, which measured 3-10 %
  // faster from S = 2048 on (b16 s2048 h12, b4 s4096 h16, b1 s16384 h8) - but at 229
  // VGPRs only two wavefronts fit a SIMD, so the 256-query blocks must fill both block
  // slots of every CU, and at S = 512 or 1024 prologue and epilogue of the fewer, larger
  // blocks cost more than the loop gains (b32 s512 h12: 9 % slower).
  const bool wideBlocks = dHead == 64 && !causal && S >= 2048 &&
                          (int64_t)B * H * ((S + 255) / 256) >= 2 * (int64_t)deviceComputeUnits();
  if (wideBlocks) launch<T, 64, 2, false>(qkv, seqlens, cuSeqlens, out, B, S, H, dHead, scale, causal, stream);
  else if (dHead == 64) launch<T, 64, 1, false>(qkv, seqlens, cuSeqlens, out, B, S, H, dHead, scale, causal, stream);
  else if (dHead == 128) launch<T, 128, 1, false>(qkv, seqlens, cuSeqlens, out, B, S, H, dHead, scale, causal, stream);
  else if (dHead == 256) launch<T, 256, 1, false>(qkv, seqlens, cuSeqlens, out, B, S, H, dHead, scale, causal, stream);
  // Sizes in between go in classes, each without the matrix steps that only filler would feed.  The lines lie where a step of 16 or 32
  // saves most at sizes in use (us, the whole geometry / the class: 32 of 64 20.6 / 16.2 at b15 s934 h4, 80 of 128 83.6 / 66.9 at b9 s1351 h8, 160 of
  // 256 111 / 82 at b8 s535 h32; over 150 launches 32: 0.87 of the time, 40: 0.96, 72 and 80: 0.93, 96: 0.94, 144 and 160: 0.87).
  else if (dHead <= 32) launch<T, 64, 1, true, 32>(qkv, seqlens, cuSeqlens, out, B, S, H, dHead, scale, causal, stream);
  else if (dHead <= 48) launch<T, 64, 1, true, 48>(qkv, seqlens, cuSeqlens, out, B, S, H, dHead, scale, causal, stream);
  else if (dHead < 64) launch<T, 64, 1, true>(qkv, seqlens, cuSeqlens, out, B, S, H, dHead, scale, causal, stream);
  else if (dHead <= 80) launch<T, 128, 1, true, 80>(qkv, seqlens, cuSeqlens, out, B, S, H, dHead, scale, causal, stream);
  else if (dHead <= 96) launch<T, 128, 1, true, 96>(qkv, seqlens, cuSeqlens, out, B, S, H, dHead, scale, causal, stream);
  else if (dHead < 128) launch<T, 128, 1, true>(qkv, seqlens, cuSeqlens, out, B, S, H, dHead, scale, causal, stream);
  else if (dHead <= 160) launch<T, 256, 1, true, 160>(qkv, seqlens, cuSeqlens, out, B, S, H, dHead, scale, causal, stream);
  else launch<T, 256, 1, true>(qkv, seqlens, cuSeqlens, out, B, S, H, dHead, scale, causal, stream);
}

} // namespace

namespace {
void fusedMHAChecked(DType dt, const void *qkv, const int32_t *seqlens, const int32_t *cuSeqlens, void *out, int B,
                     int S, int H, int D, float scale, bool causal, hipStream_t stream) {
  if (B < 0 || S < 0 || H < 0) fail("fusedMHA: negative shape");
  // 64, 128 and 256 are the tile geometries; the other head sizes of the reference's
  // dispatcher (32, 40, 80, 144, 160; fused_multihead_attention_v2.h:4646-4673) and any
  // other multiple of 8 run in the next larger geometry with the filler masked out.
  if (D < 8 || D > 256 || D % 8) fail("fusedMHA: head_dim must be a multiple of 8 between 8 and 256");
  if (B == 0 || S == 0 || H == 0) return;
  if (!qkv || !out) fail("fusedMHA: null pointer");
  if (!aligned16(qkv) || !aligned16(out)) fail("fusedMHA: qkv and out must be 16-byte aligned");
  if (!(scale > 0.0f) || !(scale < INFINITY)) fail("fusedMHA: softmax scale must be positive and finite");
  if ((int64_t)S * 3 * H * D * 2 > 0x7fffffffLL) fail("fusedMHA: one sequence of QKV must stay below 2 GiB");
  if (dt != DType::F16 && dt != DType::BF16) fail("fusedMHA: element type must be fp16 or bf16");
  if (fusedMHASplitKeys(dt, qkv, seqlens, cuSeqlens, out, B, S, H, D, scale, causal, stream)) return;
  if (dt == DType::F16) launchForHeadDim<_Float16>(qkv, seqlens, cuSeqlens, out, B, S, H, D, scale, causal, stream);
  else launchForHeadDim<bf16_t>(qkv, seqlens, cuSeqlens, out, B, S, H, D, scale, causal, stream);
}
} // namespace

void fusedMHA(DType dt, const void *qkv, const int32_t *seqlens, void *out, int B, int S, int H,
              int D, float scale, bool causal, hipStream_t stream) {
  fusedMHAChecked(dt, qkv, seqlens, nullptr, out, B, S, H, D, scale, causal, stream);
}

void fusedMHACuSeqlens(DType dt, const void *qkv, const int32_t *cuSeqlens, void *out, int B, int maxS, int H,
                       int D, float scale, bool causal, hipStream_t stream) {
  if (!cuSeqlens && B > 0 && maxS > 0 && H > 0) fail("fusedMHA: cu_seqlens is null");
  fusedMHAChecked(dt, qkv, nullptr, cuSeqlens, out, B, maxS, H, D, scale, causal, stream);
}

} // namespace mgpu
