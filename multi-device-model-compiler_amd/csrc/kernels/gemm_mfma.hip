// fp16 / bf16 GEMM with the bias, activation and residual epilogue fused, on
// gfx950 MFMA: out[M,N] = act(in[M,K] . W[K,N] + bias[N]) (+ residual[M,N]).
//
// One of the ways mgpuMatmulEx<half> (lib/Kernels/GPU/Ops.cu:134-234) is
// served; gemm.cpp has the others and the rule that chooses.  This file has the launcher for 128-row tiles: at most one a
// CU go to gemm_round.hip, more of them to gemm_wide.hip; the kernel below takes what is too shallow for those two (gemmMfmaShallow),
// several tiles a CU of fewer than 128 rows, and sizes beyond the other two's limits (gemmMfmaKernel).
//
// Work decomposition.  A 256-thread block (4 wavefronts) owns a 128 x 128 output
// tile (wavefronts 2 x 2, each 64 x 64 as 2 x 2 accumulators of 32 x 32) or a
// 128 x 96 one (wavefronts 4 x 1, each 32 x 96 as 3 accumulators); the launcher
// takes the width that loads the busiest CU least (768 columns are 6 tiles of
// 128 - 192 tiles at M = 4096, a quarter of the CUs idle - or 8 of 96 - 256
// tiles, one per CU).  The reduction runs in steps of 32: per step an 8 KiB
// slice of the input (128 rows of 64 bytes) and a slice of the weight (32 rows
// at a 256-byte pitch) travel HBM -> LDS directly (global_load_lds, 16 bytes per
// lane) into a ring of three stages, two steps in flight behind the one
// consumed; three blocks share a CU (48 KiB of LDS, < 128 VGPRs).
//
// MFMA formulation: the transposed product out^T[n, m] = W^T[n, k] . in^T[k, m],
//   A operand = W^T: the weight slice sits in LDS row-major as in memory
//     ([k][n], n contiguous); ds_read_b64_tr_b16 hands lane (n = l % 32) the
//     four k of its column, two reads per operand;
//   B operand = in^T: lane (m = l % 32) reads 16 contiguous bytes of its row.
// so that an accumulator register group holds four consecutive n of one row m:
// bias, activation and residual are applied on 8-byte pieces of output rows,
// and the tile is then transposed through LDS so that every store instruction
// writes whole 128-byte runs of output rows.  Both slices are stored unpadded
// (the direct loads fill 1 KiB of consecutive LDS per instruction) with an XOR
// swizzle on the 16-byte chunk index that keeps both operand reads free of
// bank conflicts.
//
// Shapes: K a multiple of 32, 16-byte aligned operands, and M a multiple of 128, N
// of 128 or 96 or - RAGGED below - any M and N a multiple of 8.  gemm.cpp gives the
// rest to gemm_ksplit or the library.
#include "common.hpp"
#include "mfma.hpp"
#include "mgpu_ops_internal.hpp"
#include "types.hpp"

namespace mgpu {

namespace {

constexpr int kBM = 128;       // rows of an output tile
constexpr int kBK = 32;        // reduction step
constexpr int kRing = 3;       // LDS ring depth
constexpr int kWRow = 256;     // LDS pitch of a weight-slice row, bytes (128 columns, of which NB * 32 are loaded)

// Chunk swizzles: the 16-byte chunk c of a row is kept at chunk c ^ swz(row).
__host__ __device__ constexpr int aSwz(int row) { return (row >> 2) & 3; }        // 4 chunks per row
__host__ __device__ constexpr int wSwz(int row) { return (row & 3) << 2; } // 16 chunks per row

// T: element type; ACT: epilogue activation; NB: tile width in 32-column blocks (4 or 3).
//
// RAGGED: M is no multiple of 128 or N none of the tile width.  The tiles cover the shape; rows and
// columns past the end are loaded from the last ones and not stored.
template <typename T, int ACT, int NB, bool RAGGED>
__global__ __launch_bounds__(256, 3) void gemm_mfma_kernel(const uint16_t *__restrict__ in,
                                                                        const uint16_t *__restrict__ weight,
                                                                        const uint16_t *__restrict__ bias,
                                                                        const uint16_t *residual, uint16_t *out, int N,
                                                                        int K, int tilesN, int tilesM, int M_) {
  using M = Mma<T>;
  using v8 = typename M::v8;
  using v4 = typename M::v4;
  static_assert(NB == 4 || NB == 3, "tile geometry");
  constexpr int kBN = 32 * NB;
  constexpr int kSlice = 256 * kBK;                  // bytes of an input slice, and of a weight slice at full pitch
  constexpr int kARow = kBK * 2;                     // bytes per row of the input slice
  constexpr int NC = 2, NL = 2;                      // per reduction step: MFMA k-steps; load instructions a wavefront and slice
  constexpr int CPR = kBK / 8, RPI = 64 / CPR;       // input slice: chunks per row, rows per load instruction
  constexpr int WN = NB == 4 ? 2 : 1, WM = 4 / WN;   // wavefront grid over the tile: 2 x 2 or 4 x 1
  constexpr int MB = 4 / WM, NBW = NB / WN;          // 32 x 32 accumulators per wavefront: MB x NBW = 2 x 2 or 1 x 3
  constexpr int kOutStride = 32 * NBW + 4;           // staging row stride of a wavefront's part, in elements

  // Ring of kRing stages, each an input slice followed by a weight slice;
  // reused as the output staging area at the end.
  constexpr int kLds = kRing * 2 * kSlice;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[kLds];
  static_assert(4 * 32 * MB * kOutStride * 2 <= kLds, "output staging must fit in the ring");

  // Tile order.  A contiguous run of work items goes to each of the 8 XCDs
  // (consecutive block ids are dealt round-robin to the XCDs), and consecutive
  // work items walk down kGroup rows of tiles before stepping one column, so
  // that the ~96 blocks resident on an XCD form a compact patch of tiles: the
  // slices they load per step are then few (8 input + 12 weight slices instead
  // of 2 + 64 for a row-major sweep of a wide matrix) and hit in that XCD's L2.
  constexpr int kGroup = 8;
  // (the grid is tilesM x tilesN blocks; both are explicit arguments - fourteen dwords in all,
  // what the command processor preloads into SGPRs - rather than gridDim, a kernarg-segment load)
  const int nblk = tilesM * tilesN;
  const int bid = blockIdx.x;
  const int wid = (nblk % 8 == 0) ? (bid % 8) * (nblk / 8) + bid / 8 : bid;
  const int perGroup = kGroup * tilesN;
  const int firstM = (wid / perGroup) * kGroup;
  const int groupRows = tilesM - firstM < kGroup ? tilesM - firstM : kGroup;
  const int inGroup = wid % perGroup;
  const int m0 = (firstM + inGroup % groupRows) * kBM;
  const int n0 = (inGroup / groupRows) * kBN;

  const int tid = threadIdx.x;
  const int lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int l32 = lane % 32;
  const int hl = lane / 32;
  const int wm = wave / WN, wn = wave % WN; // the wavefront's part of the tile

  // ---- slice movers: HBM -> LDS, 16 bytes per lane ----------------------------
  // One wavefront instruction fills 1 KiB: RPI rows of the input slice or 4 rows
  // of the weight slice; every wavefront moves a quarter of both.  In a 96-column
  // tile the lanes that would fetch the chunks beyond column 95 fetch a chunk of
  // the tile again instead: it lands in the unread tail of the 256-byte pitch.
  // (Masking those lanes off would put the load under divergent control flow,
  // where its scalar operands are no longer scalar to the compiler.)
  const char *abase = reinterpret_cast<const char *>(in) + (size_t)m0 * K * 2;
  const char *wbase = reinterpret_cast<const char *>(weight) + (size_t)n0 * 2;
  const int nk = K / kBK; // reduction steps
  const int rowsLeft = RAGGED ? M_ - m0 : kBM; // rows of the tile that exist
  auto memRow = [&](int row) { return RAGGED && row >= rowsLeft ? rowsLeft - 1 : row; };
  uint32_t aoff[NL], woff[NL];
#pragma unroll
  for (int i = 0; i < NL; i++) {
    const int arow = RPI * (NL * wave + i) + lane / CPR;
    aoff[i] = (uint32_t)memRow(arow) * (uint32_t)K * 2u + (uint32_t)(((lane % CPR) ^ aSwz(arow)) * 16);
    const int wrow = 4 * (NL * wave + i) + lane / 16;
    int wchunk = (lane % 16) ^ wSwz(wrow);
    if (wchunk >= 4 * NB) wchunk -= 4;
    if (RAGGED && n0 + 8 * wchunk >= N) wchunk = (N - 8 - n0) / 8;
    woff[i] = (uint32_t)wrow * (uint32_t)N * 2u + (uint32_t)(wchunk * 16);
  }
  // (2 * NL loads per stage and wavefront, counted by hand)
  const uint32_t ldsBase = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) unsigned char *)smem);
  auto issueStage = [&](int kt) {
    const uint32_t adst = ldsBase + (uint32_t)((kt % kRing) * (2 * kSlice) + (NL * wave) * 1024);
    const uint32_t wdst = adst + kSlice;
    const char *ag = abase + (size_t)kt * kARow;
    const char *wg = wbase + (size_t)kt * kBK * N * 2;
#pragma unroll
    for (int i = 0; i < NL; i++) {
      ldsLoad16(aoff[i], ag, adst + i * 1024);
      ldsLoad16(woff[i], wg, wdst + i * 1024);
    }
  };

#pragma unroll
  for (int t = 0; t < kRing - 1; t++)
    if (t < nk) issueStage(t);

  // ---- operand addresses inside a stage ---------------------------------------
  // in^T: lane (row 32*MB*wm + 32mb + l32, k chunk 2c + hl) reads 16 bytes.
  uint32_t afrag[MB][NC];
#pragma unroll
  for (int mb = 0; mb < MB; mb++)
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const int row = wm * (32 * MB) + 32 * mb + l32;
      afrag[mb][c] = (uint32_t)(row * kARow + (((2 * c + hl) ^ aSwz(row)) * 16));
    }
  // W^T: as a source of the transposing read, lane L of a 16-lane group g points
  // at k row 8*hl + L/4 (+ 16c, + 4 for the upper k-slots) and the four columns
  // n = 32nb + 16*(g%2) + 4*(L%4) .. +3.
  uint32_t wfrag[NBW]; // relative to the weight slice
  {
    const int g = lane / 16, L = lane % 16, r = L % 4, j = L / 4;
#pragma unroll
    for (int nb = 0; nb < NBW; nb++) {
      const int chunk = (4 * (NBW * wn + nb) + 2 * (g % 2) + r / 2) ^ wSwz(j);
      wfrag[nb] = (uint32_t)((8 * hl + j) * kWRow + chunk * 16 + 8 * (r % 2));
    }
  }

  f32x16 acc[NBW][MB]; // [nb][mb]: rows n, columns m
#pragma unroll
  for (int nb = 0; nb < NBW; nb++)
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[nb][mb][i] = 0.0f;

  for (int kt = 0; kt < nk; kt++) {
    // The loads of stage kt (and of nothing later) must have landed; the barrier
    // makes every wavefront's share visible and says that everybody is done
    // with stage kt-1, which the next load overwrites.
    if (kt + 1 < nk) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (kt + kRing - 1 < nk) issueStage(kt + kRing - 1);
    const uint32_t aBase = ldsBase + (uint32_t)((kt % kRing) * (2 * kSlice)); // LDS addresses of this step's input rows and weight slice
    const uint32_t wBase = aBase + kSlice;

#pragma unroll
    for (int c = 0; c < NC; c++) {
      v8 b[MB], a[NBW];
#pragma unroll
      for (int mb = 0; mb < MB; mb++)
        b[mb] = *reinterpret_cast<const v8 __attribute__((address_space(3))) *>((const lds_u8 *)(uintptr_t)(aBase + afrag[mb][c]));
#pragma unroll
      for (int nb = 0; nb < NBW; nb++) {
        const lds_u8 *p = (const lds_u8 *)(uintptr_t)(wBase + wfrag[nb]) + 16 * c * kWRow;
        const v4 lo = M::readTr(p);             // k-slots 0..3
        const v4 hi = M::readTr(p + 4 * kWRow); // k-slots 4..7
        a[nb] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
#pragma unroll
      for (int nb = 0; nb < NBW; nb++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) acc[nb][mb] = M::run(a[nb], b[mb], acc[nb][mb]);
    }
  }

  // ---- epilogue: bias, activation, residual; transpose through LDS; store ------
  __syncthreads(); // every wavefront is done reading the slices
  uint16_t *stage = reinterpret_cast<uint16_t *>(smem) + wave * (32 * MB * kOutStride);
  const int mw = m0 + wm * (32 * MB), nw = n0 + wn * (32 * NBW); // origin of the wavefront's part
  // All bias pieces of the part first, then per 32-column block all of its
  // residual pieces, so that the loads of a batch are in flight together.
  v4 braw[NBW][4];
#pragma unroll
  for (int nb = 0; nb < NBW; nb++)
#pragma unroll
    for (int g = 0; g < 4; g++)
#pragma unroll
      for (int i = 0; i < 4; i++) braw[nb][g][i] = M::narrow(0.0f);
  if (bias) {
#pragma unroll
    for (int nb = 0; nb < NBW; nb++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int n = nw + 32 * nb + 8 * g + 4 * hl;
        braw[nb][g] = *reinterpret_cast<const v4 *>(bias + (RAGGED && n >= N ? N - 4 : n));
      }
  }
#pragma unroll
  for (int nb = 0; nb < NBW; nb++) {
    v4 rraw[4][MB];
#pragma unroll
    for (int g = 0; g < 4; g++)
#pragma unroll
      for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int i = 0; i < 4; i++) rraw[g][mb][i] = M::narrow(0.0f);
    if (residual) {
#pragma unroll
      for (int g = 0; g < 4; g++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
          const int n = nw + 32 * nb + 8 * g + 4 * hl;
          rraw[g][mb] = *reinterpret_cast<const v4 *>(residual + (size_t)(m0 + memRow(mw - m0 + 32 * mb + l32)) * N +
                                                      (RAGGED && n >= N ? N - 4 : n));
        }
    }
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const int nloc = 32 * nb + 8 * g + 4 * hl; // four consecutive columns of the part
#pragma unroll
      for (int mb = 0; mb < MB; mb++) {
        const int mloc = 32 * mb + l32;
        float x[4];
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = acc[nb][mb][4 * g + i] + M::widen(braw[nb][g][i]);
        if (ACT == ACT_RELU) {
#pragma unroll
          for (int i = 0; i < 4; i++) x[i] = x[i] > 0.0f ? x[i] : 0.0f;
        } else if (ACT == ACT_GELU) {
#pragma unroll
          for (int i = 0; i < 4; i++) x[i] = M::gelu(x[i]);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] += M::widen(rraw[g][mb][i]);
        v4 o;
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] = M::narrow(x[i]);
        *reinterpret_cast<v4 *>(&stage[mloc * kOutStride + nloc]) = o;
      }
    }
  }
  // Each wavefront reads back only what it wrote: no block barrier needed, the
  // LDS accesses of one wavefront are ordered.
  constexpr int kOutChunks = 4 * NBW; // 16-byte chunks per row of the part
#pragma unroll
  for (int it = 0; it < 32 * MB * kOutChunks / 64; it++) {
    const int chunk = it * 64 + lane;
    const int r = chunk / kOutChunks, cidx = chunk % kOutChunks;
    // 8-byte LDS reads: the staging stride is 8-byte but not 16-byte aligned
    const u32x2 lo = *reinterpret_cast<const u32x2 *>(&stage[r * kOutStride + cidx * 8]);
    const u32x2 hi = *reinterpret_cast<const u32x2 *>(&stage[r * kOutStride + cidx * 8 + 4]);
    const u32x4 val = {lo[0], lo[1], hi[0], hi[1]};
    if (RAGGED && (mw + r >= M_ || nw + cidx * 8 >= N)) continue;
    *reinterpret_cast<u32x4 *>(out + (size_t)(mw + r) * N + nw + cidx * 8) = val;
  }
}

template <typename T, int NB, bool RAGGED>
void launchAct(const uint16_t *a, const uint16_t *w, const uint16_t *b, const uint16_t *r, uint16_t *o, int64_t M,
               int64_t N, int64_t K, int act, hipStream_t stream) {
  const int tilesN = (int)((N + 32 * NB - 1) / (32 * NB)), tilesM = (int)((M + kBM - 1) / kBM);
  const dim3 grid((unsigned)(tilesM * tilesN)), block(256);
  if (act == ACT_GELU)
    launchKernel(gemm_mfma_kernel<T, ACT_GELU, NB, RAGGED>, grid, block, stream, a, w, b, r, o, (int)N, (int)K, tilesN, tilesM, (int)M);
  else if (act == ACT_RELU)
    launchKernel(gemm_mfma_kernel<T, ACT_RELU, NB, RAGGED>, grid, block, stream, a, w, b, r, o, (int)N, (int)K, tilesN, tilesM, (int)M);
  else
    launchKernel(gemm_mfma_kernel<T, ACT_NONE, NB, RAGGED>, grid, block, stream, a, w, b, r, o, (int)N, (int)K, tilesN, tilesM, (int)M);
}
template <typename T, int NB>
void launchTile(const uint16_t *a, const uint16_t *w, const uint16_t *b, const uint16_t *r, uint16_t *o, int64_t M,
                int64_t N, int64_t K, int act, hipStream_t stream) {
  if (M % kBM || N % (32 * NB)) launchAct<T, NB, true>(a, w, b, r, o, M, N, K, act, stream);
  else launchAct<T, NB, false>(a, w, b, r, o, M, N, K, act, stream);
}

// Tile width: the one under which the busiest CU carries the fewest columns
// (tiles are dealt evenly, so that CU holds ceil(tiles / CUs) of them); 128 on
// a tie.
int tileWidth(int64_t M, int64_t N) {
  const int64_t cus = numComputeUnits();
  auto load = [&](int64_t width) { return ((M + kBM - 1) / kBM * ((N + width - 1) / width) + cus - 1) / cus * width; };
  return load(96) < load(128) ? 96 : 128;
}

template <typename T>
void launch(const void *in, const void *weight, const void *bias, const void *residual, void *out, int64_t M,
            int64_t N, int64_t K, int act, hipStream_t stream) {
  const auto *a = static_cast<const uint16_t *>(in);
  const auto *w = static_cast<const uint16_t *>(weight);
  const auto *b = static_cast<const uint16_t *>(bias);
  const auto *r = static_cast<const uint16_t *>(residual);
  auto *o = static_cast<uint16_t *>(out);
  const DType dt = std::is_same<T, _Float16>::value ? DType::F16 : DType::BF16;
  int width;
  const GemmKernel kernel = gemmMfmaKernel(dt, in, weight, bias, residual, out, M, N, K, act, &width);
  if (kernel == GemmKernel::Round) return gemmRound(dt, in, weight, bias, residual, out, M, N, K, act, width, stream);
  if (kernel == GemmKernel::Wide) return gemmWide(dt, in, weight, bias, residual, out, M, N, K, act, width, stream);
  if (width == 96) launchTile<T, 3>(a, w, b, r, o, M, N, K, act, stream);
  else launchTile<T, 4>(a, w, b, r, o, M, N, K, act, stream);
  MGPU_CHECK_LAUNCH("gemm_mfma_kernel");
}

} // namespace

bool gemmMfmaSupports(DType dt, const void *in, const void *weight, const void *bias, const void *residual,
                      const void *out, int64_t M, int64_t N, int64_t K) {
  if (dt != DType::F16 && dt != DType::BF16) return false;
  if (M <= 0 || N <= 0 || K <= 0 || M % kBM || (N % 128 && N % 96) || K % 32) return false;
  // 32-bit lane offsets inside a slice; fewer than 2^24 tiles, of 256 threads, in a grid dimension of fewer than 2^32
  // (which keeps the rows below 2^31)
  if (K > (1 << 20) || N > (1 << 20) || M / kBM > 0xffffff / (N / 96)) return false;
  if (!aligned16(in) || !aligned16(weight) || !aligned16(out)) return false;
  if (bias && (reinterpret_cast<uintptr_t>(bias) & 7u)) return false;
  if (residual && !aligned16(residual)) return false;
  return true;
}

bool gemmMfmaSupportsRagged(DType dt, const void *in, const void *weight, const void *bias, const void *residual,
                            const void *out, int64_t M, int64_t N, int64_t K) {
  if (N % 8) return false;
  const int64_t m = (M + kBM - 1) / kBM * kBM, n = (N + 127) / 128 * 128; // the tiles that cover the shape
  return gemmMfmaSupports(dt, in, weight, bias, residual, out, m, n, K);
}

// Is the kernel above ahead of gemm_round in one round (gemmMfmaShallow has the times)?
static bool shallowRound(int64_t N, int64_t K, bool hasResidual) {
  const bool halfStep = K % 64 == 32;
  return K % 32 == 0 && (N % 64 == 0 ? halfStep && K <= 96 && !hasResidual : K <= 64 || (halfStep && K <= 160));
}

// One tile per CU: gemm_round, fitted to 600 shapes (4 % rms, 14 % at worst; with it and gemm_ksplit's estimate the choice
// between the two is 0.3 % behind the best of them, the library and gemm_wide, whose tiles it never pays to have less than one
// round of).  Several: what overlaps of the operand bytes at 52 GB/s a CU behind 5 us of start and end.
// A shallow round without a GELU: the kernel above, ahead of a second round of gemm_ksplit's tiles and, 32 deep, of one of 64 x 64 (us,
// gemm_ksplit / it: 768 x 1152 x 32 3.85 / 3.39, 26 x 18240 x 32 4.7 / 3.8, 1 x 23568 x 96 4.45 / 3.8).
double gemmMfmaCost(int64_t M, int64_t N, int64_t K, int act, bool hasResidual) {
  const int64_t cus = numComputeUnits(), width = tileWidth(M, N), tiles = (M + kBM - 1) / kBM * ((N + width - 1) / width);
  const double bytes = (double)(kBM + width) * 2.0 * (double)K, full = (double)tiles / (double)cus;
  if (tiles <= cus && act != ACT_GELU && shallowRound(N, K, hasResidual)) return 2.0 + 0.0125 * (double)K;
  if (tiles <= cus) return 3.2 + 1.14 * full + bytes * (11.4e-6 + 2e-6 * full) + (act == ACT_GELU ? 1.4 : 0.0);
  return 5.0 + full * bytes / 52e3;
}

int gemmRoundWidth(DType dt, const void *in, const void *weight, const void *bias, const void *residual, const void *out, int64_t M, int64_t N,
                   int64_t K) {
  if (K % 8 || K * N >= int64_t(1) << 30 || !gemmMfmaSupportsRagged(dt, in, weight, bias, residual, out, M, N, (K + 31) / 32 * 32)) return 0;
  const int width = tileWidth(M, N);
  return (M + kBM - 1) / kBM * ((N + width - 1) / width) <= numComputeUnits() ? width : 0;
}

// The tile width and estimated us of gemmMfmaPartialF16 without what its planes cost (gemmPartialPlan has that); no width where
// its blocks are more than one round of the CUs.
static int partialWidth(int64_t M, int64_t N, int parts) {
  const int64_t tilesM = (M + kBM - 1) / kBM * parts;
  return tilesM * ((N + 95) / 96) <= numComputeUnits() ? 96 : tilesM * ((N + 127) / 128) <= numComputeUnits() ? 128 : 0;
}

double gemmMfmaPartialCost(int64_t M, int64_t N, int64_t K, int parts) {
  const int width = partialWidth(M, N, parts);
  return width && K % 64 == 0 ? 3.05 + (double)(kBM + width) * 2.0 * (double)K / parts * 11.3e-6 : 1e30;
}

void gemmMfmaPartialF16(const void *in, const void *weight, float *planes, int64_t M, int64_t N, int64_t K, int parts, hipStream_t stream) {
  const int width = partialWidth(M, N, parts);
  if (!gemmMfmaSupportsRagged(DType::F16, in, weight, nullptr, nullptr, planes, M, N, K) || !width || K % 64 || K / 64 < parts)
    fail("gemmMfmaPartial: internal dispatch error");
  gemmRoundPartialF16(in, weight, planes, M, N, K, width, parts, stream);
}

// Where the kernel above is ahead of gemm_round and gemm_wide although they go (us, they / this kernel): a product so shallow that their
// rings never fill, or that they fill up to a step of 64.  One round of tiles: rows that are no whole lines up to 64 deep, or 96 or 160
// (1395 x 648 x 32 4.1 / 3.6; they take 1.13 times as long at 32 on average, 1.06 at 64, 1.09 at 96, 1.07 at 160, but 1.00 at 128 and 1.01 at
// 224); whole lines at 32 and 96 (1.09, 1.03), not with a residual, which gemm_round asks for earlier (0.97, 0.93).  More rounds, up to
// 256 deep: by the estimates, this kernel's fitted to 1500 products (7.5 % rms, so that it has to win by 4 %; by 10 with a GELU up to two
// rounds, by nothing beyond, where gemm_wide's one block a CU exposes a GELU's wait each round): 5504 x 3552 x 96 15.0 / 12.7.  Of 1250
// such products it takes 191, which become 9 % faster on average (27 slower by more than 3 %, the worst 1.14 times as long).
bool gemmMfmaShallow(int64_t M, int64_t N, int64_t K, int act, bool hasResidual) {
  const int64_t cus = numComputeUnits(), width = tileWidth(M, N), tiles = (M + kBM - 1) / kBM * ((N + width - 1) / width);
  const bool wholeLines = N % 64 == 0;
  if (tiles <= cus) return shallowRound(N, K, hasResidual);
  if (K % 32 || K > 256 || M < kBM) return false;
  const double each = 0.9 + 0.0107 * (double)K + (act == ACT_GELU ? 1.45 : 0.0) + (hasResidual ? (wholeLines ? 1.6 : 1.25) : 0.0) + (wholeLines ? 0.0 : 0.15);
  double wide;
  (void)gemmWideBest(M, N, K, act, hasResidual, &wide);
  const double ahead = act != ACT_GELU ? 1.04 : tiles > 2 * cus ? 1.0 : 1.1;
  return ahead * (3.6 + (double)tiles * (double)width / (128.0 * (double)cus) * each) < wide;
}

// Which kernel runs a product here, and the width of its tiles: gemm_round when no CU gets a second tile, otherwise gemm_wide, each
// where it goes, and the kernel above where neither does or it is ahead.  The kernel above also where gemm_wide's tiles of 256 rows would be three
// quarters empty, or half and a GELU's wait exposed at one block a CU (us, gemm_wide / this kernel, with a GELU: 1 x 65536 x 256 16.9
// / 11.4, 32 x 33024 x 512 15.8 / 12.1, 127 x 65536 x 512 23.7 / 19.0; without: 32 x 65536 x 128 6.7 / 6.0, 100 x 33024 x 96 6.1 / 5.7,
// but 100 x 40000 x 128 6.0 / 6.8 and 127 x 33024 x 256 8.1 / 9.1).
GemmKernel gemmMfmaKernel(DType dt, const void *in, const void *weight, const void *bias, const void *residual, const void *out, int64_t M,
                          int64_t N, int64_t K, int act, int *width) {
  *width = tileWidth(M, N);
  if (gemmMfmaShallow(M, N, K, act, residual != nullptr)) return GemmKernel::Mfma;
  if ((M + kBM - 1) / kBM * ((N + *width - 1) / *width) <= numComputeUnits() && (K % 64 == 0 || K * N < int64_t(1) << 30))
    return GemmKernel::Round;
  const bool tooFewRows = M < kBM && (act == ACT_GELU || M <= 64 || K < 128);
  if (tooFewRows || !gemmWideSupports(dt, in, weight, bias, residual, out, M, N, K)) return GemmKernel::Mfma;
  double cost;
  *width = gemmWideBest(M, N, K, act, residual != nullptr, &cost);
  return GemmKernel::Wide;
}

void gemmMfmaRagged(DType dt, const void *in, const void *weight, const void *bias, const void *residual, void *out,
                    int64_t M, int64_t N, int64_t K, int act, hipStream_t stream) {
  if (!gemmMfmaSupportsRagged(dt, in, weight, bias, residual, out, M, N, K))
    fail("gemmMfma: shape, type or alignment not supported by the hand-written kernel");
  if (dt == DType::F16)
    launch<_Float16>(in, weight, bias, residual, out, M, N, K, act, stream);
  else
    launch<bf16_t>(in, weight, bias, residual, out, M, N, K, act, stream);
}

void gemmMfma(DType dt, const void *in, const void *weight, const void *bias, const void *residual, void *out,
              int64_t M, int64_t N, int64_t K, int act, hipStream_t stream) {
  if (!gemmMfmaSupports(dt, in, weight, bias, residual, out, M, N, K))
    fail("gemmMfma: shape, type or alignment not supported by the hand-written kernel");
  if (act != ACT_NONE && residual) fail("gemmMfma: an activation cannot be combined with a residual");
  if (dt == DType::F16)
    launch<_Float16>(in, weight, bias, residual, out, M, N, K, act, stream);
  else
    launch<bf16_t>(in, weight, bias, residual, out, M, N, K, act, stream);
}

} // namespace mgpu
