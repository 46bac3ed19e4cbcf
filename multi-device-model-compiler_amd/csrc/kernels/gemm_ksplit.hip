// fp16 / bf16 GEMM for few tiles: out[M,N] = act(in[M,K] . W[K,N] + bias[N]) (+ residual[M,N]), any
// M, N and K multiples of 8; the weight as the ABI gives it or K-major ([N, K]).
//
// A serving-size GEMM (one request of 77 tokens against 768 x 3072 weights) is a handful of output
// tiles: tiled like a large one it leaves most CUs idle behind a long serial reduction.  Here a block
// owns a small tile, 32 MB x 32 NB, and its KS wavefronts split the REDUCTION: wavefront ks takes a
// contiguous share of the k range for the whole tile, so every operand byte is still read once per
// block, and nothing is shared between wavefronts until the end - no barrier in the loop.  Each
// wavefront streams its operands HBM -> LDS (global_load_lds, 16 bytes per lane) into a ring of its
// own, chunks of 32 k, RING of them in flight; the partial tiles meet in LDS, where all threads
// sum them and apply bias, activation and residual in fp32 (one rounding).
//
// MFMA formulation and operand reads are those of gemm_mfma.hip: the transposed product
// out^T[n, m] = W^T[n, k] . in^T[k, m] with W^T through the transposing LDS read.
//
// Result::Planes: the blocks of grid row y take the y-th share of the reduction and write their fp32 sums to plane y of `out`
// (float [parts][M][N]; partial_sums.hip adds the planes up and has the epilogue).  Result::F32: the rounded result, widened (the
// bits of a cast behind the kernel).
#include "common.hpp"
#include "mfma.hpp"
#include "mgpu_ops_internal.hpp"
#include "types.hpp"

namespace mgpu {

namespace {

typedef float float4v __attribute__((ext_vector_type(4)));

constexpr int kSplit = 8; // wavefronts of a block

enum class Result { Half, Planes, F32 };
template <typename T, int ACT, int MB, int NB, int RING, bool KMAJOR, Result RESULT = Result::Half>
__global__ __launch_bounds__(64 * kSplit, 1) void gemm_ksplit_kernel(const uint16_t *__restrict__ in, const uint16_t *__restrict__ weight,
                                                                 const uint16_t *__restrict__ bias, ResidualOrShare<RESULT == Result::Planes> residual, uint16_t *out,
                                                                 int M, int N, int K, int tilesM, int nblk) {
  using Mm = Mma<T>;
  using v8 = typename Mm::v8;
  using v4 = typename Mm::v4;
  constexpr int KS = kSplit, BM = 32 * MB, BN = 32 * NB;
  constexpr int kX = 2048 * MB, kW = 2048 * NB;      // bytes of a chunk's input rows (64 bytes each) and weight rows (64 NB bytes)
  constexpr int kStage = kX + kW;
  constexpr int ND = 2 * (MB + NB);                  // 1 KiB load instructions per chunk
  constexpr int kPart = 8 * 528;                     // bytes of a 32 x 32 partial tile (padded against bank conflicts)
  constexpr int kWave = RING * kStage > MB * NB * kPart ? RING * kStage : (MB * NB * kPart + 1023) / 1024 * 1024;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[KS * kWave];

  // Tile order: a contiguous run of tiles goes to each XCD, tiles of one column of W next to each other, so
  // that each weight column is read into one XCD's L2 only.
  const int bid = blockIdx.x, xcd = bid % 8, q8 = nblk / 8, r8 = nblk % 8;
  const int wid = xcd * q8 + (xcd < r8 ? xcd : r8) + bid / 8;
  const int m0 = (wid % tilesM) * BM, n0 = (wid / tilesM) * BN;

  const int tid = threadIdx.x, lane = tid % 64;
  const int ks = __builtin_amdgcn_readfirstlane(tid / 64);
  const int l32 = lane % 32, hl = lane / 32;

  int chunks = (K + 31) / 32, firstChunk = 0;
  if constexpr (RESULT == Result::Planes) {
    firstChunk = divide(chunks * (int)blockIdx.y, residual);
    chunks = divide(chunks * ((int)blockIdx.y + 1), residual) - firstChunk;
  }
  const int c0 = firstChunk + chunks * ks / KS, c1 = firstChunk + chunks * (ks + 1) / KS;

  // ---- movers: per instruction 16 input rows of 64 bytes, or 1 KiB of weight rows.  Rows and columns past
  // the end are clamped to the last ones (their products are not stored), k past the end likewise (those
  // operands are zeroed in registers).
  const char *xbase = reinterpret_cast<const char *>(in) + (size_t)m0 * K * 2;
  const char *wbase = reinterpret_cast<const char *>(weight);
  int xrow[2 * MB], xk[2 * MB];
#pragma unroll
  for (int i = 0; i < 2 * MB; i++) {
    const int row = 16 * i + lane / 4;
    xrow[i] = (row < M - m0 ? row : M - 1 - m0);
    xk[i] = 8 * ((lane % 4) ^ ((row >> 2) & 3)); // first k of the 16-byte piece (XOR swizzle against bank conflicts)
  }
  constexpr int WPR = 4 * NB, WRI = 64 / WPR; // 16-byte pieces per weight row, rows per instruction
  auto wSwz = [](int row) { return NB == 2 ? ((row >> 1) & 1) << 2 : 0; };
  // A K-major weight (KMAJOR: [N, K]) is moved and read like the input rows.
  int wk[2 * NB], wcol[2 * NB]; // first k and column of the 16-byte piece
#pragma unroll
  for (int i = 0; i < 2 * NB; i++) {
    if (KMAJOR) {
      const int row = 16 * i + lane / 4;
      wcol[i] = n0 + row < N ? row : N - 1 - n0;
      wk[i] = 8 * ((lane % 4) ^ ((row >> 2) & 3));
      continue;
    }
    wk[i] = WRI * i + lane / WPR;
    const int col = n0 + 8 * ((lane % WPR) ^ wSwz(wk[i]));
    wcol[i] = col < N ? col : N - 8;
  }
  const uint32_t ldsBase = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) unsigned char *)smem) + (uint32_t)ks * kWave;
  // (inline assembly: completion is tracked by hand, see gemm_mfma.hip)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  auto dma16 = [&](uint32_t voffset, const char *sbase, uint32_t ldsAddr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(voffset), "s"(sbase), "s"(ldsAddr)
                 : "memory", "m0");
  };
#pragma clang diagnostic pop
  auto issue = [&](int c, int stage) {
    const uint32_t at = ldsBase + (uint32_t)stage * kStage;
    const int k0 = 32 * c;
    const char *wrow = wbase + (KMAJOR ? (size_t)n0 * K : (size_t)k0 * N) * 2;
#pragma unroll
    for (int i = 0; i < 2 * MB; i++) {
      const int k = k0 + xk[i] < K ? k0 + xk[i] : K - 8;
      dma16((uint32_t)(xrow[i] * K + k) * 2u, xbase, at + i * 1024);
    }
#pragma unroll
    for (int i = 0; i < 2 * NB; i++) {
      if (KMAJOR) {
        const int k = k0 + wk[i] < K ? k0 + wk[i] : K - 8;
        dma16((uint32_t)(wcol[i] * K + k) * 2u, wrow, at + kX + i * 1024);
      } else {
        const int k = k0 + wk[i] < K ? wk[i] : K - 1 - k0;
        dma16((uint32_t)(k * N + wcol[i]) * 2u, wrow, at + kX + i * 1024);
      }
    }
  };
#pragma unroll
  for (int r = 0; r < RING; r++)
    if (c0 + r < c1) issue(c0 + r, r);

  // ---- operand addresses inside a stage (see gemm_mfma.hip)
  uint32_t xfrag[MB][2], wfrag[NB], wfragK[NB][2];
#pragma unroll
  for (int mb = 0; mb < MB; mb++)
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const int row = 32 * mb + l32;
      xfrag[mb][c] = (uint32_t)(row * 64 + (((2 * c + hl) ^ ((row >> 2) & 3)) * 16));
    }
#pragma unroll
  for (int nb = 0; nb < NB; nb++) {
    const int g = lane / 16, L = lane % 16, r = L % 4, j = L / 4;
    const int row = 8 * hl + j;
    const int piece = (4 * nb + 2 * (g % 2) + r / 2) ^ wSwz(row);
    wfrag[nb] = (uint32_t)(kX + row * (64 * NB) + piece * 16 + 8 * (r % 2));
#pragma unroll
    for (int c = 0; c < 2; c++)
      wfragK[nb][c] = (uint32_t)(kX + (32 * nb + l32) * 64 + (((2 * c + hl) ^ (((32 * nb + l32) >> 2) & 3)) * 16));
  }

  f32x16 acc[NB][MB];
#pragma unroll
  for (int nb = 0; nb < NB; nb++)
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[nb][mb][i] = 0.0f;

  int stage = 0;
  for (int c = c0; c < c1; c++) {
    // chunk c has landed; up to RING - 1 later ones may fly
    const int later = c1 - 1 - c;
    if (RING > 3 && later >= 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * ND) : "memory");
    else if (RING > 2 && later >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * ND) : "memory");
    else if (later >= 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(ND) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const uint32_t at = ldsBase + (uint32_t)stage * kStage;
    auto step = [&](int s, bool masked) {
      v8 a[NB], b[MB];
#pragma unroll
      for (int mb = 0; mb < MB; mb++)
        b[mb] = *reinterpret_cast<const v8 __attribute__((address_space(3))) *>((const lds_u8 *)(uintptr_t)(at + xfrag[mb][s]));
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        if (KMAJOR) {
          a[nb] = *reinterpret_cast<const v8 __attribute__((address_space(3))) *>((const lds_u8 *)(uintptr_t)(at + wfragK[nb][s]));
          continue;
        }
        const lds_u8 *p = (const lds_u8 *)(uintptr_t)(at + wfrag[nb]) + 16 * s * (64 * NB);
        const v4 lo = Mm::readTr(p);
        const v4 hi = Mm::readTr(p + 4 * (64 * NB));
        a[nb] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
      if (masked) { // the last eight k of K = 16 n + 8: the upper lane half's slots are past the end
        const v8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int mb = 0; mb < MB; mb++) b[mb] = hl ? zero : b[mb];
#pragma unroll
        for (int nb = 0; nb < NB; nb++) a[nb] = hl ? zero : a[nb];
      }
#pragma unroll
      for (int nb = 0; nb < NB; nb++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) acc[nb][mb] = Mm::run(a[nb], b[mb], acc[nb][mb]);
    };
    const int left = K - 32 * c; // (uniform)
    if (left >= 32) {
      step(0, false);
      step(1, false);
    } else {
      step(0, left < 16);
      if (left > 16) step(1, true);
    }
    if (c + RING < c1) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the reads of this stage are done before it is overwritten
      issue(c + RING, stage);
    }
    stage = stage == RING - 1 ? 0 : stage + 1;
  }

  // ---- partial tiles to LDS (each wavefront into its own ring's place), sum, epilogue ----------
  // 16-byte piece (register group g, lane half hl, row m) at (2 g + hl) * 528 + 16 m.
#pragma unroll
  for (int nb = 0; nb < NB; nb++)
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
      for (int g = 0; g < 4; g++)
        *reinterpret_cast<float4v *>(smem + ks * kWave + (nb * MB + mb) * kPart + (2 * g + hl) * 528 + l32 * 16) =
            float4v{acc[nb][mb][4 * g], acc[nb][mb][4 * g + 1], acc[nb][mb][4 * g + 2], acc[nb][mb][4 * g + 3]};
  __syncthreads();
  // A thread sums four consecutive columns of one row: eight (sixteen) threads a row, 64 (128) bytes of output.
  constexpr int QN = BN / 4, UNITS = BM * QN;
#pragma unroll
  for (int u0 = 0; u0 < UNITS; u0 += 64 * KS) {
    const int u = u0 + tid;
    if (UNITS % (64 * KS) && u >= UNITS) break;
    const int mrow = u / QN, q = u % QN;
    const int m = m0 + mrow, n = n0 + 4 * q;
    if (m >= M || n >= N) continue;
    const unsigned char *part = smem + ((q / 8) * MB + mrow / 32) * kPart + (q % 8) * 528 + (mrow % 32) * 16;
    float4v x = *reinterpret_cast<const float4v *>(part);
#pragma unroll
    for (int s = 1; s < KS; s++) x += *reinterpret_cast<const float4v *>(part + s * kWave);
    if (RESULT == Result::Planes) {
      *reinterpret_cast<float4v *>(reinterpret_cast<float *>(out) + ((size_t)blockIdx.y * M + m) * N + n) = x;
      continue;
    }
    if (bias) {
      const v4 b = *reinterpret_cast<const v4 *>(bias + n);
#pragma unroll
      for (int i = 0; i < 4; i++) x[i] += Mm::widen(b[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      if (ACT == ACT_RELU) x[i] = x[i] > 0.0f ? x[i] : 0.0f;
      if (ACT == ACT_GELU) x[i] = Mm::gelu(x[i]);
    }
    if constexpr (RESULT != Result::Planes) {
      if (residual) {
        const v4 r = *reinterpret_cast<const v4 *>(residual + (size_t)m * N + n);
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] += Mm::widen(r[i]);
      }
    }
    v4 o;
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = Mm::narrow(x[i]);
    if (RESULT == Result::F32) {
#pragma unroll
      for (int i = 0; i < 4; i++) x[i] = Mm::widen(o[i]);
      *reinterpret_cast<float4v *>(reinterpret_cast<float *>(out) + (size_t)m * N + n) = x;
      continue;
    }
    *reinterpret_cast<v4 *>(out + (size_t)m * N + n) = o;
  }
}

template <typename T, int MB, int NB, int RING, bool KMAJOR>
void launchTile(const uint16_t *a, const uint16_t *w, const uint16_t *b, const uint16_t *r, uint16_t *o, int64_t M, int64_t N, int64_t K,
                int act, hipStream_t stream) {
  const int tilesM = (int)((M + 32 * MB - 1) / (32 * MB)), tilesN = (int)((N + 32 * NB - 1) / (32 * NB));
  const int nblk = tilesM * tilesN;
  const dim3 grid((unsigned)nblk), block(64 * kSplit);
  if (act == ACT_GELU)
    launchKernel(gemm_ksplit_kernel<T, ACT_GELU, MB, NB, RING, KMAJOR>, grid, block, stream, a, w, b, r, o, (int)M, (int)N, (int)K, tilesM, nblk);
  else if (act == ACT_RELU)
    launchKernel(gemm_ksplit_kernel<T, ACT_RELU, MB, NB, RING, KMAJOR>, grid, block, stream, a, w, b, r, o, (int)M, (int)N, (int)K, tilesM, nblk);
  else
    launchKernel(gemm_ksplit_kernel<T, ACT_NONE, MB, NB, RING, KMAJOR>, grid, block, stream, a, w, b, r, o, (int)M, (int)N, (int)K, tilesM, nblk);
}

template <typename T, bool KMAJOR>
void launch(const void *in, const void *weight, const void *bias, const void *residual, void *out, int64_t M, int64_t N, int64_t K, int act,
            KSplitTile tile, hipStream_t stream) {
  const auto *a = static_cast<const uint16_t *>(in);
  const auto *w = static_cast<const uint16_t *>(weight);
  const auto *b = static_cast<const uint16_t *>(bias);
  const auto *r = static_cast<const uint16_t *>(residual);
  auto *o = static_cast<uint16_t *>(out);
  if (tile == KSplitTile::T32x32) launchTile<T, 1, 1, 4, KMAJOR>(a, w, b, r, o, M, N, K, act, stream);
  else if (tile == KSplitTile::T32x64) launchTile<T, 1, 2, 3, KMAJOR>(a, w, b, r, o, M, N, K, act, stream);
  else launchTile<T, 2, 2, 2, KMAJOR>(a, w, b, r, o, M, N, K, act, stream);
  MGPU_CHECK_LAUNCH("gemm_ksplit_kernel");
}

} // namespace

// us of the variant on a shape, up to a constant all hand-written variants share: one tile per CU and round,
// a fixed part (first loads, partial sums, epilogue) and the tile's operand bytes at the 55 GB/s a CU pulls.
// (77 x 2304 x 768 32 x 32: 4.5 us; 77 x 3072 x 768 + GELU 32 x 64: 5.3; 300 x 3072 x 768 + GELU 64 x 64: 8.2.)
KSplitTile gemmKSplitBest(int64_t M, int64_t N, int64_t K, int act, double *cost, int parts) {
  auto costOf = [&](int bm, int bn, double fixed) {
    const int64_t tiles = (M + bm - 1) / bm * ((N + bn - 1) / bn) * parts;
    const int64_t rounds = (tiles + numComputeUnits() - 1) / numComputeUnits();
    return (double)rounds * (fixed + (double)(bm + bn) * 2.0 * (double)K / parts / 55e3);
  };
  const double c[3] = {costOf(32, 32, 1.8), costOf(32, 64, 1.9), costOf(64, 64, act == ACT_GELU ? 3.6 : 2.4)};
  const int best = c[0] <= c[1] && c[0] <= c[2] ? 0 : c[1] <= c[2] ? 1 : 2;
  *cost = c[best];
  return best == 0 ? KSplitTile::T32x32 : best == 1 ? KSplitTile::T32x64 : KSplitTile::T64x64;
}

bool gemmKSplitSupports(DType dt, const void *in, const void *weight, const void *bias, const void *residual, const void *out, int64_t M,
                        int64_t N, int64_t K) {
  if (dt != DType::F16 && dt != DType::BF16) return false;
  if (M <= 0 || N <= 0 || K <= 0 || N % 8 || K % 8) return false;
  // 32-bit offsets from a tile's first row (64 rows of the input, 32 of the weight), 31-bit tile counts
  if (K > (1 << 20) || N > (1 << 20) || M > (1 << 30) || (M + 31) / 32 * ((N + 31) / 32) > 0x7fffffffLL) return false;
  if (!aligned16(in) || !aligned16(weight) || !aligned16(out)) return false;
  if (bias && (reinterpret_cast<uintptr_t>(bias) & 7u)) return false;
  return !residual || aligned16(residual);
}

void gemmKSplit(DType dt, const void *in, const void *weight, const void *bias, const void *residual, void *out, int64_t M, int64_t N,
                int64_t K, int act, KSplitTile tile, bool weightKMajor, hipStream_t stream) {
  if (dt == DType::F16) {
    if (weightKMajor) launch<_Float16, true>(in, weight, bias, residual, out, M, N, K, act, tile, stream);
    else launch<_Float16, false>(in, weight, bias, residual, out, M, N, K, act, tile, stream);
  } else {
    if (weightKMajor) launch<bf16_t, true>(in, weight, bias, residual, out, M, N, K, act, tile, stream);
    else launch<bf16_t, false>(in, weight, bias, residual, out, M, N, K, act, tile, stream);
  }
}

void gemmKSplitPartialF16(const void *in, const void *weight, float *planes, int64_t M, int64_t N, int64_t K, KSplitTile tile, int parts,
                          hipStream_t stream) {
  if (!gemmKSplitSupports(DType::F16, in, weight, nullptr, nullptr, planes, M, N, K)) fail("gemmKSplitPartial: internal dispatch error");
  const auto *a = static_cast<const uint16_t *>(in);
  const auto *w = static_cast<const uint16_t *>(weight);
  auto *o = reinterpret_cast<uint16_t *>(planes);
  const PartShare share = partShare(parts);
  const int bm = tile == KSplitTile::T64x64 ? 64 : 32, bn = tile == KSplitTile::T32x32 ? 32 : 64;
  const int tilesM = (int)((M + bm - 1) / bm), nblk = tilesM * (int)((N + bn - 1) / bn);
  const dim3 grid((unsigned)nblk, (unsigned)parts), block(64 * kSplit);
  const int m = (int)M, n = (int)N, k = (int)K;
  if (tile == KSplitTile::T32x32)
    launchKernel(gemm_ksplit_kernel<_Float16, ACT_NONE, 1, 1, 4, false, Result::Planes>, grid, block, stream, a, w, nullptr, share, o, m, n, k, tilesM, nblk);
  else if (tile == KSplitTile::T32x64)
    launchKernel(gemm_ksplit_kernel<_Float16, ACT_NONE, 1, 2, 3, false, Result::Planes>, grid, block, stream, a, w, nullptr, share, o, m, n, k, tilesM, nblk);
  else
    launchKernel(gemm_ksplit_kernel<_Float16, ACT_NONE, 2, 2, 2, false, Result::Planes>, grid, block, stream, a, w, nullptr, share, o, m, n, k, tilesM, nblk);
  MGPU_CHECK_LAUNCH("gemm_ksplit_kernel");
}

namespace {
template <bool KMAJOR>
void launchToF32(const void *in, const void *weight, const void *bias, const void *residual, float *out, int64_t M, int64_t N, int64_t K,
                 KSplitTile tile, hipStream_t stream) {
  auto go = [&](auto *kernel, int bm, int bn) {
    const int tilesM = (int)((M + bm - 1) / bm), nblk = tilesM * (int)((N + bn - 1) / bn);
    launchKernel(kernel, dim3((unsigned)nblk), dim3(64 * kSplit), stream, static_cast<const uint16_t *>(in), static_cast<const uint16_t *>(weight),
        static_cast<const uint16_t *>(bias), static_cast<const uint16_t *>(residual), reinterpret_cast<uint16_t *>(out), (int)M, (int)N, (int)K, tilesM, nblk);
  };
  if (tile == KSplitTile::T32x32) go(gemm_ksplit_kernel<_Float16, ACT_NONE, 1, 1, 4, KMAJOR, Result::F32>, 32, 32);
  else if (tile == KSplitTile::T32x64) go(gemm_ksplit_kernel<_Float16, ACT_NONE, 1, 2, 3, KMAJOR, Result::F32>, 32, 64);
  else go(gemm_ksplit_kernel<_Float16, ACT_NONE, 2, 2, 2, KMAJOR, Result::F32>, 64, 64);
  MGPU_CHECK_LAUNCH("gemm_ksplit_kernel");
}
} // namespace

void gemmKSplitResidualF32(const void *in, const void *weight, const void *bias, const void *residual, float *out, int64_t M, int64_t N,
                           int64_t K, KSplitTile tile, bool weightKMajor, hipStream_t stream) {
  if (weightKMajor) launchToF32<true>(in, weight, bias, residual, out, M, N, K, tile, stream);
  else launchToF32<false>(in, weight, bias, residual, out, M, N, K, tile, stream);
}

} // namespace mgpu
