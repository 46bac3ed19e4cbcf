// fp16 / bf16 GEMM on 128-row tiles, at most one per CU: out[M,N] = act(in[M,K] . W[K,N] + bias[N]) (+ residual[M,N]).
//
// The kernel for products of some 60 to 256 tiles of 128 x 128 or 128 x 96 (gemm_mfma.hip's launcher and gemm.cpp choose):
// the second FFN product and the projection of a transformer layer at a few thousand tokens.  Formulation as in
// gemm_mfma.hip, schedule as in gemm_wide.hip, where the reasons stand: loads spread between the matrix instructions,
// operands double-buffered in registers across the barrier.
//
// What bounds it: the loads.  A tile this small has 57 (128 x 96) or 64 FLOP a byte, and a CU pulls 35 bytes a clock from
// L2 whatever is in flight: 800 clocks for a step of 64 of the reduction, against 384 of matrix instructions.  So everything
// else has to fit under them: the whole LDS is one ring of five steps, four of them in flight (112 or 128 KB); eight
// wavefronts, of which 0-3 and 4-7 cover the tile in the same way and take the lower and the upper half of every step
// (a step's barrier comes half as often as with four covering it once, and the LDS reads of a part of 64 x 64 are the fewest
// per matrix instruction); and both sets of wavefronts share the epilogue, each with half of every accumulator.
//
// Shapes: any M, N a multiple of 8 (tiles overhang the shape: rows and columns past the end are loaded from the last ones
// and not stored), K a multiple of 8 (filled up to one of 64 with zeros; planes: of 64), 16-byte aligned operands.
#include "common.hpp"
#include "mfma.hpp"
#include "mgpu_ops_internal.hpp"
#include "types.hpp"

namespace mgpu {

namespace {

typedef float float4v __attribute__((ext_vector_type(4)));

constexpr int kBM = 128;
constexpr int kThreads = 512;

// Chunk swizzles of the LDS rows (see gemm_wide.hip); rows of the weight are 256 or 192 bytes, and 192 spread by themselves.
__host__ __device__ constexpr int aSwz(int row) { return (row >> 1) & 7; }
template <int NB> __host__ __device__ constexpr int wSwz(int row) { return NB == 4 ? (row & 3) << 2 : 0; }

// ACT: the activation, or one of
constexpr int kResidual = 3; // + residual in its place
constexpr int kPartial = 4;  // the blocks of grid row y take the y-th share of the reduction and write their fp32 sums to
                             // plane y of `out` (float [parts][M][N]; partial_sums.hip adds them up and has the epilogue)
constexpr int kResidualF32 = 5; // + residual, the rounded result widened to fp32 (the bits of a cast behind the kernel)
template <typename T, int ACT, int NB, bool RAGGED>
__global__ __launch_bounds__(kThreads, 2) void gemm_round_kernel(const uint16_t *__restrict__ in, const uint16_t *__restrict__ weight,
                                                                 const uint16_t *__restrict__ bias, ResidualOrShare<ACT == kPartial> residual, uint16_t *out,
                                                                 int N, int K, int tilesN, int tilesM, int M_) {
  using M = Mma<T>;
  using v8 = typename M::v8;
  using v4 = typename M::v4;
  constexpr bool RESIDUAL = ACT == kResidual || ACT == kResidualF32;
  constexpr int BN = 32 * NB;
  constexpr int kA = kBM * 128, kW = 64 * BN * 2, kStage = kA + kW; // a step of 64: 16 KiB of input rows, 16 or 12 of the weight
  constexpr int kRing = 5, kAhead = kRing - 1;
  constexpr int WN = NB == 4 ? 2 : 1, WM = 4 / WN; // wavefront grid over the tile: 2 x 2 or 4 x 1
  constexpr int MB = 4 / WM, NBW = NB / WN;        // 32 x 32 accumulators of a wavefront: 2 x 2 or 1 x 3
  constexpr int CPR = BN / 8;                      // 16-byte chunks of a weight row
  constexpr int kOutStride = 32 * NBW + 4;         // staging row stride of a part, in elements
  constexpr int kStaging = 4 * 32 * MB * kOutStride * 2;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[kRing * kStage];
  static_assert(kStaging + 8 * NBW * MB * 8 * 64 * 4 <= kRing * kStage, "output staging and exchange must fit the ring");

  // Tile order as in gemm_wide.hip: a run of tiles for each XCD, down kGroup rows before the next column.
  constexpr int kGroup = 8;
  const int nblk = tilesM * tilesN, xcd = blockIdx.x % 8, share = nblk / 8, extra = nblk % 8;
  const int wid = xcd * share + (xcd < extra ? xcd : extra) + (int)blockIdx.x / 8;
  const int perGroup = kGroup * tilesN;
  const int firstM = (wid / perGroup) * kGroup;
  const int groupRows = tilesM - firstM < kGroup ? tilesM - firstM : kGroup;
  const int inGroup = wid % perGroup;
  const int m0 = (firstM + inGroup % groupRows) * kBM;
  const int n0 = (inGroup / groupRows) * BN;

  const int tid = threadIdx.x, lane = tid % 64, l32 = lane % 32, hl = lane / 32;
  const int mover = __builtin_amdgcn_readfirstlane(tid / 64);
  const int khalf = mover / 4, wave = mover % 4;
  const int wm = wave / WN, wn = wave % WN; // the part of the tile that wavefronts `wave` and `wave` + 4 share

  // ---- loads: two instructions of input rows and two (NB 3: one and a half) of the weight a wavefront and step ------
  const char *ag = reinterpret_cast<const char *>(in) + (size_t)m0 * K * 2;
  const char *wg = reinterpret_cast<const char *>(weight) + (size_t)n0 * 2;
  int steps = RAGGED ? (K + 63) / 64 : K / 64;
  if constexpr (ACT == kPartial) {
    const int first = divide(steps * (int)blockIdx.y, residual);
    steps = divide(steps * ((int)blockIdx.y + 1), residual) - first;
    ag += (size_t)first * 128;
    wg += (size_t)first * 128 * N;
  }
  const int rowsLeft = M_ - m0;
  uint32_t aoff[2], woff[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int row = 8 * (2 * mover + i) + lane / 8, memRow = row >= rowsLeft ? rowsLeft - 1 : row;
    aoff[i] = (uint32_t)memRow * (uint32_t)K * 2u + (uint32_t)(((lane % 8) ^ aSwz(row)) * 16);
    const int c = mover * (kW / 128) + 64 * i + lane; // chunk of the slice (past its end only in lanes that are off)
    const int wrow = (c / CPR) % 64;
    int chunk = (c % CPR) ^ wSwz<NB>(wrow);
    if (n0 + 8 * chunk >= N) chunk = (N - 8 - n0) / 8;
    woff[i] = (uint32_t)wrow * (uint32_t)N * 2u + (uint32_t)(chunk * 16);
  }
  const uint32_t ldsBase = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) unsigned char *)smem);
  uint32_t fill = 0; // offset of the ring slot filled next
  // RAGGED: K ends inside the last step, whose loads past it arrive as zeros (see gemm_wide.hip).
  i32x4 abuf{}, wbuf{};
  int k0 = 0; // first column and row of the step loaded next
  if (RAGGED) {
    abuf = ldsBuffer(ag, (uint32_t)(rowsLeft < kBM ? rowsLeft : kBM) * (uint32_t)K * 2u);
    wbuf = ldsBuffer(wg, ((uint32_t)K * (uint32_t)N - (uint32_t)n0) * 2u);
  }
  auto issueW = [&](int i) {
    const uint32_t dst = ldsBase + fill + (uint32_t)(kA + mover * (kW / 8) + i * 1024);
    if (RAGGED && NB == 3 && i == 1) ldsLoad16LowerLanes(woff[i], wbuf, (uint32_t)k0 * (uint32_t)N * 2u, dst);
    else if (RAGGED) ldsLoad16(woff[i], wbuf, (uint32_t)k0 * (uint32_t)N * 2u, dst);
    else if (NB == 3 && i == 1) ldsLoad16LowerLanes(woff[i], wg, dst);
    else ldsLoad16(woff[i], wg, dst);
  };
  auto issueA = [&](int i) {
    const uint32_t dst = ldsBase + fill + (uint32_t)((2 * mover + i) * 1024);
    if (!RAGGED) return ldsLoad16(aoff[i], ag, dst);
    const int column = ((lane % 8) ^ aSwz(8 * i + lane / 8)) * 8; // (rows 16 apart have the same swizzle)
    ldsLoad16(column < K - k0 ? aoff[i] : kPastBuffer, abuf, (uint32_t)k0 * 2u, dst);
  };
  auto nextIssue = [&]() {
    k0 += 64;
    ag += 128;
    wg += (size_t)N * 128;
    fill = fill == (kRing - 1) * kStage ? 0 : fill + kStage;
  };

  // ---- operands ---------------------------------------------------------------------
  // k-step c of this half of a step: chunks 4 khalf + 2c + hl of the input rows, weight rows 32 khalf + 16c + ...
  uint32_t afrag[2], wfrag[NBW];
#pragma unroll
  for (int c = 0; c < 2; c++) {
    const int row = wm * (32 * MB) + l32;
    afrag[c] = ldsBase + (uint32_t)(row * 128 + (((4 * khalf + 2 * c + hl) ^ aSwz(row)) * 16));
  }
  {
    const int g = lane / 16, L = lane % 16, r = L % 4, j = L / 4;
#pragma unroll
    for (int nb = 0; nb < NBW; nb++) {
      const int chunk = (4 * (NBW * wn + nb) + 2 * (g % 2) + r / 2) ^ wSwz<NB>(j);
      wfrag[nb] = ldsBase + (uint32_t)(kA + (32 * khalf + 8 * hl + j) * (BN * 2) + chunk * 16 + 8 * (r % 2));
    }
  }
  struct Operands {
    v8 b[MB], a[NBW];
  };
  Operands o0{}, o1{};
  f32x16 acc[NBW][MB]; // [nb][mb]: rows n, columns m
  uint32_t use = 0;    // offset of the step in use
  auto nextStep = [&]() { use = use == (kRing - 1) * kStage ? 0 : use + kStage; };
  auto readB = [&](Operands &o, int c) {
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
      o.b[mb] = *reinterpret_cast<const v8 __attribute__((address_space(3))) *>((const lds_u8 *)(uintptr_t)(afrag[c] + use) + mb * 4096);
  };
  auto readA = [&](Operands &o, int c, int nb) {
    const lds_u8 *p = (const lds_u8 *)(uintptr_t)(wfrag[nb] + use) + 16 * c * (BN * 2);
    const v4 lo = M::readTr(p);
    const v4 hi = M::readTr(p + 4 * (BN * 2));
    o.a[nb] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto readAll = [&](Operands &o, int c) {
    readB(o, c);
#pragma unroll
    for (int nb = 0; nb < NBW; nb++) readA(o, c, nb);
  };
  auto multiplyAll = [&](const Operands &o) {
#pragma unroll
    for (int j = 0; j < NBW * MB; j++) acc[j / MB][j % MB] = M::run(o.a[j / MB], o.b[j % MB], acc[j / MB][j % MB]);
  };
  // One k-step: the matrix instructions on `u`; between them the reads of the k-step after it and two loads.
  auto kStep = [&](const Operands &u, Operands &f, int c, int load) { // load: 0 none, 1 weight, 2 input
#pragma unroll
    for (int j = 0; j < NBW * MB; j++) {
      if (j == 0) readB(f, c);
      if (j == 0) readA(f, c, 0);
      if (j == 1) {
        readA(f, c, 1);
        if (load == 1) issueW(0);
        if (load == 2) issueA(0);
      }
      if (j == 2) {
        if (NBW == 3) readA(f, c, NBW - 1);
        if (load == 1) issueW(1);
        if (load == 2) issueA(1);
      }
      __builtin_amdgcn_sched_barrier(0);
      acc[j / MB][j % MB] = M::run(u.a[j / MB], u.b[j % MB], acc[j / MB][j % MB]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#define MGPU_WAIT_AND_BARRIER(n) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(n) : "memory")

  // ---- main loop ----------------------------------------------------------------------
  // The bias, by the lower half only, through the ring slot that is filled last into the accumulators (see gemm_wide.hip).
  const bool biased = ACT != kPartial && bias != nullptr && khalf == 0;
  const uint32_t biasAt = ldsBase + (uint32_t)((kRing - 1) * kStage + wave * 256);
  if (biased) {
    const int n = n0 + wn * (32 * NBW) + 2 * lane;
    ldsLoad4((uint32_t)(n < N ? n : N - 2) * 2u, reinterpret_cast<const char *>(bias), biasAt);
  }
#pragma unroll
  for (int s = 0; s < kAhead; s++)
    if (s < steps) {
      issueW(0), issueW(1), issueA(0), issueA(1);
      nextIssue();
    }
  if (biased) {
    if (steps >= kAhead) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * kAhead) : "memory"); // all but the bias may be in flight
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
#pragma unroll
  for (int nb = 0; nb < NBW; nb++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      v4 b = {};
      if (biased) b = *reinterpret_cast<const v4 __attribute__((address_space(3))) *>((const lds_u8 *)(uintptr_t)(biasAt + 8 * hl) + 64 * nb + 16 * g);
#pragma unroll
      for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int i = 0; i < 4; i++) acc[nb][mb][4 * g + i] = M::widen(b[i]);
    }
  if (steps >= kAhead) {
    // Behind the barrier of step s, group s of the loads: the weight rows of step s + 4 between the matrix instructions of
    // the first k-step, its input rows - behind the barrier of s + 1 - between those of the second.  A step needs the group
    // four before it: two whole groups and one weight share may still be in flight.
    MGPU_WAIT_AND_BARRIER(12);
    readAll(o0, 0);
    __builtin_amdgcn_sched_barrier(0);
    for (int s = 0; s < steps - kAhead; s++) {
      kStep(o0, o1, 1, 1);
      nextStep();
      MGPU_WAIT_AND_BARRIER(10);
      kStep(o1, o0, 0, 2);
      nextIssue();
    }
    kStep(o0, o1, 1, 0);
    nextStep();
    MGPU_WAIT_AND_BARRIER(8);
    kStep(o1, o0, 0, 0);
    kStep(o0, o1, 1, 0);
    nextStep();
    MGPU_WAIT_AND_BARRIER(4);
    kStep(o1, o0, 0, 0);
    kStep(o0, o1, 1, 0);
    nextStep();
    MGPU_WAIT_AND_BARRIER(0);
    kStep(o1, o0, 0, 0);
  } else { // fewer steps than the ring: all of them at once
    MGPU_WAIT_AND_BARRIER(0);
    for (int s = 0; s < steps; s++) {
      readAll(o0, 0);
      if (s + 1 < steps) {
        readAll(o1, 1);
        multiplyAll(o0);
        multiplyAll(o1);
        nextStep();
      }
    }
  }

  // ---- epilogue -------------------------------------------------------------------------
  const int mw = m0 + wm * (32 * MB), nw = n0 + wn * (32 * NBW); // origin of the part
  const int rowsHere = M_ - mw < 32 * MB ? M_ - mw : 32 * MB;
  const int partBytes = rowsHere > 0 && nw < N ? (rowsHere * N - nw) * 2 : 0; // from the part's origin to the end of its last row
  const size_t partAt = (size_t)mw * N + nw;
  // The part as 16-byte chunks of its rows, shared by the part's two wavefronts; columns past the end point beyond it.
  constexpr int kChunks = 4 * NBW, kMine = 32 * MB * kChunks / 128;
  uint16_t *stage = reinterpret_cast<uint16_t *>(smem) + wave * (32 * MB * kOutStride);
  auto chunkRow = [&](int it) { return (it * 128 + khalf * 64 + lane) / kChunks; };
  auto chunkCol = [&](int it) { return (it * 128 + khalf * 64 + lane) % kChunks; };
  auto chunkOffset = [&](int it) { return nw + 8 * chunkCol(it) < N ? (uint32_t)(chunkRow(it) * N * 2 + chunkCol(it) * 16) : 0x40000000u; };
  u32x4 rraw[kMine];
  if constexpr (RESIDUAL) { // on its way under the last matrix instructions
    const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(residual + partAt), 0, partBytes, 0x00020000);
#pragma unroll
    for (int it = 0; it < kMine; it++) rraw[it] = __builtin_amdgcn_raw_buffer_load_b128(rows, chunkOffset(it), 0, 0);
  }
  // the last step's two k-steps
  readAll(o1, 1);
  multiplyAll(o0);
  multiplyAll(o1);
#undef MGPU_WAIT_AND_BARRIER
  __syncthreads(); // every wavefront is done reading the ring
  // Half of every accumulator goes to the part's other wavefront - the lower one finishes register groups 0 and 1, the upper
  // one 2 and 3 -, 16 bytes a lane.
  float4v *exchange = reinterpret_cast<float4v *>(smem + kStaging);
  constexpr int kSent = NBW * MB * 2;
  auto slot = [&](int from, int j) { return &exchange[(from * kSent + j) * 64 + lane]; };
#pragma unroll
  for (int nb = 0; nb < NBW; nb++)
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
      for (int g = 0; g < 2; g++) {
        float4v x;
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = khalf ? acc[nb][mb][4 * g + i] : acc[nb][mb][8 + 4 * g + i];
        *slot(mover, (nb * MB + mb) * 2 + g) = x;
      }
  if (RESIDUAL) {
#pragma unroll
    for (int it = 0; it < kMine; it++) { // (8-byte accesses: the staging stride is no multiple of 16 bytes)
      uint16_t *p = &stage[chunkRow(it) * kOutStride + 8 * chunkCol(it)];
      *reinterpret_cast<u32x2 *>(p) = u32x2{rraw[it][0], rraw[it][1]};
      *reinterpret_cast<u32x2 *>(p + 4) = u32x2{rraw[it][2], rraw[it][3]};
    }
  }
  __syncthreads();
#pragma unroll
  for (int nb = 0; nb < NBW; nb++)
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
      for (int g = 0; g < 2; g++) {
        const float4v other = *slot(mover ^ 4, (nb * MB + mb) * 2 + g);
        const int row = 32 * mb + l32, col = 32 * nb + 16 * khalf + 8 * g + 4 * hl; // four consecutive columns of the part
        float4v x;
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = (khalf ? acc[nb][mb][8 + 4 * g + i] : acc[nb][mb][4 * g + i]) + other[i];
        if (ACT == kPartial) {
          float *plane = reinterpret_cast<float *>(out) + (size_t)blockIdx.y * M_ * N;
          if (mw + row < M_ && nw + col < N) *reinterpret_cast<float4v *>(plane + (size_t)(mw + row) * N + nw + col) = x;
          continue;
        }
        uint16_t *p = &stage[row * kOutStride + col];
        if (RESIDUAL) {
          const v4 r = *reinterpret_cast<const v4 *>(p);
#pragma unroll
          for (int i = 0; i < 4; i++) x[i] += M::widen(r[i]);
        }
        if (ACT == kResidualF32) {
#pragma unroll
          for (int i = 0; i < 4; i++) x[i] = M::widen(M::narrow(x[i]));
          if (mw + row < M_ && nw + col < N) *reinterpret_cast<float4v *>(reinterpret_cast<float *>(out) + (size_t)(mw + row) * N + nw + col) = x;
          continue;
        }
        v4 o;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          if (ACT == ACT_RELU) x[i] = x[i] > 0.0f ? x[i] : 0.0f;
          if (ACT == ACT_GELU) x[i] = M::gelu(x[i]);
          o[i] = M::narrow(x[i]);
        }
        *reinterpret_cast<v4 *>(p) = o;
      }
  if (ACT == kPartial || ACT == kResidualF32) return;
  __syncthreads();
  const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(out + partAt, 0, partBytes, 0x00020000);
#pragma unroll
  for (int it = 0; it < kMine; it++) {
    const uint16_t *p = &stage[chunkRow(it) * kOutStride + 8 * chunkCol(it)];
    const u32x2 lo = *reinterpret_cast<const u32x2 *>(p);
    const u32x2 hi = *reinterpret_cast<const u32x2 *>(p + 4);
    // (as in gemm_wide.hip)
    if (N % 64) __builtin_amdgcn_raw_buffer_store_b128(u32x4{lo[0], lo[1], hi[0], hi[1]}, rows, chunkOffset(it), 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b128(u32x4{lo[0], lo[1], hi[0], hi[1]}, rows, chunkOffset(it), 0, 16);
  }
}

template <typename T, int NB, bool RAGGED>
void launch(const uint16_t *a, const uint16_t *w, const uint16_t *b, const uint16_t *r, uint16_t *o, int64_t M, int64_t N, int64_t K,
            int act, hipStream_t stream) {
  const int tilesM = (int)((M + kBM - 1) / kBM), tilesN = (int)((N + 32 * NB - 1) / (32 * NB));
  const dim3 grid((unsigned)(tilesM * tilesN)), block(kThreads);
  if (r) launchKernel(gemm_round_kernel<T, kResidual, NB, RAGGED>, grid, block, stream, a, w, b, r, o, (int)N, (int)K, tilesN, tilesM, (int)M);
  else if (act == ACT_GELU) launchKernel(gemm_round_kernel<T, ACT_GELU, NB, RAGGED>, grid, block, stream, a, w, b, r, o, (int)N, (int)K, tilesN, tilesM, (int)M);
  else if (act == ACT_RELU) launchKernel(gemm_round_kernel<T, ACT_RELU, NB, RAGGED>, grid, block, stream, a, w, b, r, o, (int)N, (int)K, tilesN, tilesM, (int)M);
  else launchKernel(gemm_round_kernel<T, ACT_NONE, NB, RAGGED>, grid, block, stream, a, w, b, r, o, (int)N, (int)K, tilesN, tilesM, (int)M);
  MGPU_CHECK_LAUNCH("gemm_round_kernel");
}

template <typename T>
void launchWidth(const void *in, const void *weight, const void *bias, const void *residual, void *out, int64_t M, int64_t N, int64_t K,
                 int act, int width, hipStream_t stream) {
  const auto *a = static_cast<const uint16_t *>(in), *w = static_cast<const uint16_t *>(weight), *b = static_cast<const uint16_t *>(bias),
             *r = static_cast<const uint16_t *>(residual);
  auto *o = static_cast<uint16_t *>(out);
  if (width == 128 && K % 64) launch<T, 4, true>(a, w, b, r, o, M, N, K, act, stream);
  else if (width == 128) launch<T, 4, false>(a, w, b, r, o, M, N, K, act, stream);
  else if (K % 64) launch<T, 3, true>(a, w, b, r, o, M, N, K, act, stream);
  else launch<T, 3, false>(a, w, b, r, o, M, N, K, act, stream);
}

} // namespace

// (The callers, gemm.cpp and gemm_mfma.hip, have checked the shape and the operands.)
void gemmRound(DType dt, const void *in, const void *weight, const void *bias, const void *residual, void *out, int64_t M, int64_t N,
               int64_t K, int act, int width, hipStream_t stream) {
  if (N % 8 || K % 8 || (K % 64 && K * N >= int64_t(1) << 30) || (act != ACT_NONE && residual) || (width != 96 && width != 128)) fail("gemmRound: internal dispatch error");
  if (dt == DType::F16) launchWidth<_Float16>(in, weight, bias, residual, out, M, N, K, act, width, stream);
  else launchWidth<bf16_t>(in, weight, bias, residual, out, M, N, K, act, width, stream);
}

void gemmRoundResidualF32(const void *in, const void *weight, const void *bias, const void *residual, float *out, int64_t M, int64_t N,
                          int64_t K, int width, hipStream_t stream) {
  if (N % 8 || K % 8 || (K % 64 && K * N >= int64_t(1) << 30) || !residual || (width != 96 && width != 128)) fail("gemmRound: internal dispatch error");
  const int tilesM = (int)((M + kBM - 1) / kBM), tilesN = (int)((N + width - 1) / width);
  auto go = [&](auto *kernel) {
    launchKernel(kernel, dim3((unsigned)(tilesM * tilesN)), dim3(kThreads), stream, static_cast<const uint16_t *>(in), static_cast<const uint16_t *>(weight),
        static_cast<const uint16_t *>(bias), static_cast<const uint16_t *>(residual), reinterpret_cast<uint16_t *>(out), (int)N, (int)K, tilesN, tilesM, (int)M);
  };
  if (width == 128 && K % 64) go(gemm_round_kernel<_Float16, kResidualF32, 4, true>);
  else if (width == 128) go(gemm_round_kernel<_Float16, kResidualF32, 4, false>);
  else if (K % 64) go(gemm_round_kernel<_Float16, kResidualF32, 3, true>);
  else go(gemm_round_kernel<_Float16, kResidualF32, 3, false>);
  MGPU_CHECK_LAUNCH("gemm_round_kernel");
}

void gemmRoundPartialF16(const void *in, const void *weight, float *planes, int64_t M, int64_t N, int64_t K, int width, int parts,
                         hipStream_t stream) {
  if (N % 8 || K % 64 || K / 64 < parts || (width != 96 && width != 128)) fail("gemmRoundPartial: internal dispatch error");
  const int tilesM = (int)((M + kBM - 1) / kBM), tilesN = (int)((N + width - 1) / width);
  const dim3 grid((unsigned)(tilesM * tilesN), (unsigned)parts), block(kThreads);
  const auto *a = static_cast<const uint16_t *>(in), *w = static_cast<const uint16_t *>(weight);
  auto *o = reinterpret_cast<uint16_t *>(planes);
  if (width == 128) launchKernel(gemm_round_kernel<_Float16, kPartial, 4, false>, grid, block, stream, a, w, nullptr, partShare(parts), o, (int)N, (int)K, tilesN, tilesM, (int)M);
  else launchKernel(gemm_round_kernel<_Float16, kPartial, 3, false>, grid, block, stream, a, w, nullptr, partShare(parts), o, (int)N, (int)K, tilesN, tilesM, (int)M);
  MGPU_CHECK_LAUNCH("gemm_round_kernel");
}

} // namespace mgpu
