// fp16 / bf16 GEMM on 256-row tiles, one block per CU: out[M,N] = act(in[M,K] . W[K,N] + bias[N]) (+ residual[M,N]).
//
// The kernel for products of many tiles (mgpuMatmulEx<half>, lib/Kernels/GPU/Ops.cu:134-234; gemm.cpp chooses).  The same
// transposed MFMA formulation as gemm_mfma.hip - out^T = W^T . in^T, so that an accumulator register group is four
// consecutive columns of one output row - on a schedule of its own.
//
// What bounds such a product, measured on 256 x 192 tiles per step of 32 of the reduction and CU, in shader clocks: the
// matrix instructions 768; the operand loads alone 717 (what a CU pulls from L2 into LDS: 35-38 bytes a clock whatever is
// in flight, so a tile must be this large for the loads to hide behind the matrix cores); the LDS reads alone 540.  A
// schedule that overlaps all three ends at the device's power limit instead: on varied operands the clock falls to
// 1.45-1.5 GHz at 880-980 clocks a step, 1.2-1.3 PFLOP/s, where all-zero operands run the same code at 2.0.  Three things
// make the overlap:
//  * one block of eight wavefronts (4 x 2, each 64 rows x BN / 2 columns) with the whole LDS: a ring of three input
//    buffers (256 rows x 64 of K each: whole 128-byte lines) and of four or five weight slices (32 of K), two buffers and
//    three or four slices in flight ahead of the one in use - over 100 KB a CU;
//  * the loads go out one at a time between the matrix instructions.  Issued together behind the barrier they fill the
//    address path (16 clocks a wavefront instruction, 44 of them a step) and every wavefront waits there with the matrix
//    cores idle: 1243 clocks a step so, 975 spread out, 4096 x 6144 x 2048 99 -> 94 us;
//  * operands are double-buffered in registers: the LDS reads of a k-step of 16 go out between the matrix instructions of
//    the one before, across the barrier.
//
// Shapes: any M, N a multiple of 8 (tiles overhang the shape: rows and columns past the end are loaded from the last ones
// and not stored), K a multiple of 8 from 72 on (filled up to a multiple of 64 with zeros), 16-byte aligned operands.
#include "common.hpp"
#include "mfma.hpp"
#include "mgpu_ops_internal.hpp"
#include "types.hpp"

#include <type_traits>

namespace mgpu {

namespace {

constexpr int kBM = 256; // rows of a tile
constexpr int kThreads = 512;

// Chunk swizzles: the 16-byte chunk c of an LDS row is kept at chunk c ^ swz(row), so that the 16 rows (input) and the 4
// rows (weight, transposing reads) of one LDS cycle lie in different banks.  Rows of the input are 128 bytes, of the
// weight BN * 2: 256, 384 or 512.
__host__ __device__ constexpr int aSwz(int row) { return (row >> 1) & 7; }
template <int BN> __host__ __device__ constexpr int wSwz(int row) { return BN == 192 ? ((row >> 1) & 1) << 2 : (row & 3) << 2; }

// ACT: the activation, or kResidual in its place.  Out: uint16_t for T's own type, or float.
constexpr int kResidual = 3;
template <typename T, int ACT, int BN, typename Out, bool RAGGED>
__global__ __launch_bounds__(kThreads, 2) void gemm_wide_kernel(const uint16_t *__restrict__ in, const uint16_t *__restrict__ weight,
                                                                const uint16_t *__restrict__ bias, const uint16_t *residual, Out *out,
                                                                int N, int K, int tilesN, int tilesM, int M_) {
  using M = Mma<T>;
  using v8 = typename M::v8;
  using v4 = typename M::v4;
  constexpr int kABuf = kBM * 128;                    // bytes of an input buffer: two steps of 32
  constexpr int kWSlice = 32 * BN * 2;                // bytes of a weight slice: one step
  constexpr int kARing = 3, kWRing = BN == 256 ? 4 : 5;
  constexpr int kWBase = kARing * kABuf;
  constexpr int kLds = kWBase + kWRing * kWSlice;     // 160, 156 or 136 KiB
  constexpr int kAhead = kWRing - 1;                  // weight slices on their way ahead of a step
  constexpr int NBW = BN / 64;                        // a wavefront's columns in blocks of 32; its rows are two blocks
  constexpr int CPR = BN / 8;                         // 16-byte chunks of a weight row
  constexpr int kOutStride = 32 * NBW + 4;            // staging row stride of a wavefront's part, in elements
  constexpr int WI = (kWSlice / 8 + 1023) / 1024;     // load instructions of a wavefront per weight slice
  constexpr bool kHalf = (kWSlice / 8) % 1024 != 0;   // the last of them by half of its lanes (BN 192)
  __shared__ __attribute__((aligned(1024))) unsigned char smem[kLds];
  static_assert(kLds <= 160 * 1024 && 8 * 64 * kOutStride * 2 <= kLds, "ring and output staging must fit the LDS");

  // Tile order: a contiguous run of tiles for each of the 8 XCDs (consecutive block ids are dealt round-robin to them),
  // whatever the number of tiles, walking down kGroup rows of tiles before stepping one column: the tiles in flight on an
  // XCD are a compact patch whose slices hit in its L2.
  constexpr int kGroup = 4;
  const int nblk = tilesM * tilesN, xcd = blockIdx.x % 8, share = nblk / 8, extra = nblk % 8;
  const int wid = xcd * share + (xcd < extra ? xcd : extra) + (int)blockIdx.x / 8;
  const int perGroup = kGroup * tilesN;
  const int firstM = (wid / perGroup) * kGroup;
  const int groupRows = tilesM - firstM < kGroup ? tilesM - firstM : kGroup;
  const int inGroup = wid % perGroup;
  const int m0 = (firstM + inGroup % groupRows) * kBM;
  const int n0 = (inGroup / groupRows) * BN;

  const int tid = threadIdx.x, lane = tid % 64, l32 = lane % 32, hl = lane / 32;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wm = wave / 2, wn = wave % 2; // the wavefront's part of the tile

  // ---- loads: L2 -> LDS, 16 bytes a lane ----------------------------------------
  const char *ag = reinterpret_cast<const char *>(in) + (size_t)m0 * K * 2;
  const char *wg = reinterpret_cast<const char *>(weight) + (size_t)n0 * 2;
  const int rowsLeft = M_ - m0;
  auto memRow = [&](int row) { return row >= rowsLeft ? rowsLeft - 1 : row; };
  uint32_t aoff[4], woff[WI];
#pragma unroll
  for (int i = 0; i < 4; i++) { // 8 rows of 128 bytes an instruction
    const int row = 8 * (4 * wave + i) + lane / 8;
    aoff[i] = (uint32_t)memRow(row) * (uint32_t)K * 2u + (uint32_t)(((lane % 8) ^ aSwz(row)) * 16);
  }
#pragma unroll
  for (int i = 0; i < WI; i++) {
    const int c = wave * (kWSlice / 128) + 64 * i + lane; // chunk of the slice (past its end only in lanes that are off)
    const int row = (c / CPR) % 32;
    int chunk = (c % CPR) ^ wSwz<BN>(row);
    if (n0 + 8 * chunk >= N) chunk = (N - 8 - n0) / 8;
    woff[i] = (uint32_t)row * (uint32_t)N * 2u + (uint32_t)(chunk * 16);
  }
  // RAGGED: K ends inside a buffer.  There the loads go through the buffer check: weight rows past the end are past the weight's
  // last, and the lanes whose chunk of an input row is past its end are pointed outside; both arrive as zeros.
  i32x4 abuf{}, wbuf{};
  int kA = 0, kW = 0; // first column of the buffer, first row of the slice filled next
  if (RAGGED) {
    abuf = ldsBuffer(ag, (uint32_t)(rowsLeft < kBM ? rowsLeft : kBM) * (uint32_t)K * 2u);
    wbuf = ldsBuffer(wg, ((uint32_t)K * (uint32_t)N - (uint32_t)n0) * 2u);
  }
  const uint32_t ldsBase = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) unsigned char *)smem);
  int aSlot = 0, wSlot = 0; // ring slots filled next
  auto issueA = [&](int i) {
    const uint32_t dst = ldsBase + (uint32_t)(aSlot * kABuf + wave * 4096 + i * 1024);
    if (!RAGGED) return ldsLoad16(aoff[i], ag, dst);
    const int column = ((lane % 8) ^ aSwz(8 * i + lane / 8)) * 8;
    ldsLoad16(column < K - kA ? aoff[i] : kPastBuffer, abuf, (uint32_t)kA * 2u, dst);
  };
  auto nextIssueA = [&]() {
    ag += 128;
    kA += 64;
    aSlot = aSlot == kARing - 1 ? 0 : aSlot + 1;
  };
  auto issueW = [&](int i) {
    const uint32_t dst = ldsBase + (uint32_t)(kWBase + wSlot * kWSlice + wave * (kWSlice / 8) + i * 1024);
    if (RAGGED) {
      const bool past = kW >= K;
      const uint32_t voff = past ? kPastBuffer : woff[i], soff = past ? 0u : (uint32_t)kW * (uint32_t)N * 2u;
      if (kHalf && i == WI - 1) ldsLoad16LowerLanes(voff, wbuf, soff, dst);
      else ldsLoad16(voff, wbuf, soff, dst);
    } else if (kHalf && i == WI - 1) ldsLoad16LowerLanes(woff[i], wg, dst);
    else ldsLoad16(woff[i], wg, dst);
  };
  auto nextIssueW = [&]() {
    wg += (size_t)N * 64;
    kW += 32;
    wSlot = wSlot == kWRing - 1 ? 0 : wSlot + 1;
  };
  auto issueSlice = [&]() {
#pragma unroll
    for (int i = 0; i < WI; i++) issueW(i);
    nextIssueW();
  };

  // ---- operands: LDS -> registers -------------------------------------------------
  // in^T: lane (row 64 wm + 32 mb + l32) reads 16 bytes, chunk 2c + hl of the buffer's 8 (c: k-step of the buffer, 0..3).
  uint32_t afrag[4];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int row = wm * 64 + l32;
    afrag[c] = ldsBase + (uint32_t)(row * 128 + (((2 * c + hl) ^ aSwz(row)) * 16));
  }
  // W^T: lane L of a 16-lane group g points at k row 8 hl + L / 4 (+ 4 for the upper k-slots) and four columns of block nb.
  uint32_t wfrag[NBW];
  {
    const int g = lane / 16, L = lane % 16, r = L % 4, j = L / 4;
#pragma unroll
    for (int nb = 0; nb < NBW; nb++) {
      const int chunk = (4 * (NBW * wn + nb) + 2 * (g % 2) + r / 2) ^ wSwz<BN>(j);
      wfrag[nb] = ldsBase + (uint32_t)(kWBase + (8 * hl + j) * (BN * 2) + chunk * 16 + 8 * (r % 2));
    }
  }
  f32x16 acc[NBW][2]; // [nb][mb]: rows n, columns m
  struct Operands {
    v8 b[2], a[NBW];
  };
  Operands o0{}, o1{};
  uint32_t aBuf = 0, wBuf = 0; // offsets of the buffer and the slice in use
  auto nextBuffer = [&]() { aBuf = aBuf == (kARing - 1) * kABuf ? 0 : aBuf + kABuf; };
  auto nextSlice = [&]() { wBuf = wBuf == (kWRing - 1) * kWSlice ? 0 : wBuf + kWSlice; };
  auto readB = [&](Operands &o, int c) {
#pragma unroll
    for (int mb = 0; mb < 2; mb++)
      o.b[mb] = *reinterpret_cast<const v8 __attribute__((address_space(3))) *>((const lds_u8 *)(uintptr_t)(afrag[c] + aBuf) + mb * 4096);
  };
  auto readA = [&](Operands &o, int half, int nb) { // half: k-step of the slice, 0 or 1
    const lds_u8 *p = (const lds_u8 *)(uintptr_t)(wfrag[nb] + wBuf) + 16 * half * (BN * 2);
    const v4 lo = M::readTr(p);
    const v4 hi = M::readTr(p + 4 * (BN * 2));
    o.a[nb] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };

  // ---- main loop --------------------------------------------------------------------
  // Step s uses slice s and half of buffer s / 2, as k-steps (s, 0) and (s, 1).  Behind the barrier of step s, when every
  // wavefront has read all of step s - 1, group s of the loads goes out: slice s + kAhead between the matrix instructions
  // of (s, 0), then - behind the barrier of s + 1 - half of buffer s / 2 + 2 between those of (s, 1).  Order of issue,
  // which the waits count on: W(s + kAhead), half A, W(s + 1 + kAhead), half A, ...; G loads a wavefront and group.
  constexpr int G = 2 + WI;
  // Loads that may still be in flight at the barrier of a step, i.e. those behind the last one it needs: for an even step
  // (slice s; the second half of buffer s / 2 from group s - 3) group s - 2 and the slice of s - 1; for an odd one what
  // followed slice s, issued kAhead groups before.  The last three steps have fewer behind them.
  constexpr int kEven = G + WI, kOdd = kAhead == 4 ? 3 * G : 2 * G;
  constexpr int kThirdLast = kAhead == 4 ? 2 + 2 * G : 2 + G + WI, kSecondLast = kAhead == 4 ? 0 : WI;
  // (lgkmcnt: this wavefront's own reads have left the slot that the next loads overwrite)
#define MGPU_WAIT_AND_BARRIER(n) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(n) : "memory")
  // One k-step: the matrix instructions on `use`; between them the operand reads of the k-step after it and the loads.
  // The fences hold each read and load at its place between two matrix instructions.
  auto kStep = [&](const Operands &use, Operands &fill, int c, int half, bool loadSlice, int loadHalfA) {
#pragma unroll
    for (int j = 0; j < 2 * NBW; j++) {
      if (j == 0) readB(fill, c);
      if (j >= 1 && j <= NBW) readA(fill, half, j - 1);
      if (j == 1) {
        if (loadSlice) issueW(0);
        if (loadHalfA >= 0) issueA(2 * loadHalfA);
      }
      if (j == (NBW == 2 ? 3 : NBW)) {
        if (loadSlice && WI == 2) issueW(1);
        if (loadHalfA >= 0) issueA(2 * loadHalfA + 1);
      }
      __builtin_amdgcn_sched_barrier(0);
      const int nb = j / 2, mb = j % 2;
      acc[nb][mb] = M::run(use.a[nb], use.b[mb], acc[nb][mb]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  const int steps = RAGGED ? (K + 63) / 64 * 2 : K / 32; // even, at least 4
  // The bias, two columns a lane, goes ahead of all other loads into a corner of the input buffer that is filled last, and
  // from there into the accumulators, while the first operands are on their way.
  const uint32_t biasAt = ldsBase + (uint32_t)(2 * kABuf + wave * 256);
  if (bias) {
    const int n = n0 + wn * (32 * NBW) + 2 * lane;
    ldsLoad4((uint32_t)(n < N ? n : N - 2) * 2u, reinterpret_cast<const char *>(bias), biasAt);
  }
  if (kAhead == 4) issueSlice();
  issueA(0), issueA(1);
  issueSlice();
  issueA(2), issueA(3);
  nextIssueA();
  issueSlice();
  issueA(0), issueA(1);
  issueSlice();
  issueA(2), issueA(3);
  nextIssueA();
  if (bias) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 + kAhead * WI) : "memory"); // all but the bias may be in flight
#pragma unroll
  for (int nb = 0; nb < NBW; nb++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      v4 b = {};
      if (bias) b = *reinterpret_cast<const v4 __attribute__((address_space(3))) *>((const lds_u8 *)(uintptr_t)(biasAt + 8 * hl) + 64 * nb + 16 * g);
#pragma unroll
      for (int i = 0; i < 4; i++) acc[nb][0][4 * g + i] = acc[nb][1][4 * g + i] = M::widen(b[i]);
    }
  MGPU_WAIT_AND_BARRIER(kEven + 2);
  readB(o0, 0);
#pragma unroll
  for (int nb = 0; nb < NBW; nb++) readA(o0, 0, nb);
  __builtin_amdgcn_sched_barrier(0);
  for (int s = 0; s < steps - 4; s += 2) {
    kStep(o0, o1, 1, 1, true, -1); // on (s, 0); reads (s, 1)
    nextIssueW();
    nextSlice();
    MGPU_WAIT_AND_BARRIER(kOdd);
    kStep(o1, o0, 2, 0, false, 0); // on (s, 1); reads (s + 1, 0)
    kStep(o0, o1, 3, 1, true, -1);
    nextIssueW();
    nextSlice();
    nextBuffer();
    MGPU_WAIT_AND_BARRIER(kEven);
    kStep(o1, o0, 0, 0, false, 1);
    nextIssueA();
  }
  // the last four steps: their loads are on the way but for the last slice where only three are kept ahead
  kStep(o0, o1, 1, 1, kAhead == 3, -1);
  nextSlice();
  MGPU_WAIT_AND_BARRIER(kThirdLast);
  kStep(o1, o0, 2, 0, false, -1);
  kStep(o0, o1, 3, 1, false, -1);
  nextSlice();
  nextBuffer();
  MGPU_WAIT_AND_BARRIER(kSecondLast);
  kStep(o1, o0, 0, 0, false, -1);
  kStep(o0, o1, 1, 1, false, -1);
  nextSlice();
  MGPU_WAIT_AND_BARRIER(0);
  // The part's rows leave - and a residual's come in - as 16-byte chunks through buffers that end with the last row;
  // lanes whose column is past the end point beyond them.  64 * kCols chunks are whole rows.
  const int mw = m0 + wm * 64, nw = n0 + wn * (32 * NBW); // origin of the part
  constexpr int kOutChunks = 4 * NBW, kCols = kOutChunks == 12 ? 3 : 1, kRowStep = 64 * kCols / kOutChunks;
  const int rowsHere = M_ - mw < 64 ? M_ - mw : 64, partBytes = rowsHere > 0 && nw < N ? (rowsHere * N - nw) * 2 : 0;
  const size_t partAt = (size_t)mw * N + nw;
  uint32_t goff[kCols];
  uint16_t *staged[kCols];
  uint16_t *stage = reinterpret_cast<uint16_t *>(smem) + wave * (64 * kOutStride);
#pragma unroll
  for (int i = 0; i < kCols; i++) {
    const int r = (64 * i + lane) / kOutChunks, c = (64 * i + lane) % kOutChunks;
    goff[i] = nw + 8 * c < N ? (uint32_t)(r * N * 2 + c * 16) : 0x40000000u;
    staged[i] = &stage[r * kOutStride + 8 * c];
  }
  u32x4 rraw[kOutChunks / 2]; // half of the part's residual
  auto loadResidual = [&](int mb) {
    const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(residual + partAt), 0, partBytes, 0x00020000);
#pragma unroll
    for (int it = 0; it < kOutChunks / 2; it++)
      rraw[it] = __builtin_amdgcn_raw_buffer_load_b128(rows, goff[it % kCols] + (uint32_t)((32 * mb + it / kCols * kRowStep) * N * 2), 0, 0);
  };
  if (ACT == kResidual) loadResidual(0);
  kStep(o1, o0, 2, 0, false, -1);
  kStep(o0, o1, 3, 1, false, -1);
#pragma unroll
  for (int j = 0; j < 2 * NBW; j++) acc[j / 2][j % 2] = M::run(o1.a[j / 2], o1.b[j % 2], acc[j / 2][j % 2]);
#undef MGPU_WAIT_AND_BARRIER

  // ---- epilogue: activation, residual; transpose through LDS; store -------------------
  // Through a staging area of the wavefront's own (the LDS accesses of one wavefront are ordered), in the layout of the
  // output's rows: a residual, asked for before the last k-steps, comes in through it and the result goes out through it.
  // One 32-row half of the part after the other, so that the first one's stores drain under the second one's arithmetic.
  // (fp32: the same area holds one half's rows, 16 * odd bytes apart.)
  __syncthreads(); // every wavefront is done reading the ring
  constexpr bool kWide = sizeof(Out) == 4;
  constexpr int kOutSize = (int)sizeof(Out), kStoreChunks = kOutChunks * kOutSize / 2, kStoreCols = kStoreChunks == 12 || kStoreChunks == 24 ? 3 : 1,
                kStoreRowStep = 64 * kStoreCols / kStoreChunks;
  const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(out + partAt, 0, partBytes / 2 * kOutSize, 0x00020000);
  float *wideStage = reinterpret_cast<float *>(stage);
  uint32_t soff[kStoreCols];
  int sat[kStoreCols];
#pragma unroll
  for (int i = 0; i < kStoreCols; i++) {
    const int r = (64 * i + lane) / kStoreChunks, c = (64 * i + lane) % kStoreChunks;
    soff[i] = nw + 16 / kOutSize * c < N ? (uint32_t)(r * N * kOutSize + c * 16) : 0x40000000u;
    sat[i] = r * kOutStride + 16 / kOutSize * c;
  }
#pragma unroll
  for (int mb = 0; mb < 2; mb++) {
    uint16_t *pieces = &stage[(32 * mb + l32) * kOutStride + 4 * hl];
    v4 r[NBW][4];
    if (ACT == kResidual) {
      if (mb == 1) loadResidual(1);
#pragma unroll
      for (int it = 0; it < kOutChunks / 2; it++) { // (8-byte accesses: the staging stride is no multiple of 16 bytes)
        uint16_t *p = staged[it % kCols] + (32 * mb + it / kCols * kRowStep) * kOutStride;
        *reinterpret_cast<u32x2 *>(p) = u32x2{rraw[it][0], rraw[it][1]};
        *reinterpret_cast<u32x2 *>(p + 4) = u32x2{rraw[it][2], rraw[it][3]};
      }
#pragma unroll
      for (int nb = 0; nb < NBW; nb++)
#pragma unroll
        for (int g = 0; g < 4; g++) r[nb][g] = *reinterpret_cast<const v4 *>(pieces + 32 * nb + 8 * g);
    }
#pragma unroll
    for (int nb = 0; nb < NBW; nb++)
#pragma unroll
      for (int g = 0; g < 4; g++) { // four consecutive columns
        v4 o;
        f32x4 wide;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float x = acc[nb][mb][4 * g + i];
          if (ACT == ACT_RELU) x = x > 0.0f ? x : 0.0f;
          if (ACT == ACT_GELU) x = M::gelu(x);
          if (ACT == kResidual) x += M::widen(r[nb][g][i]);
          if (kWide) wide[i] = x;
          else o[i] = M::narrow(x);
        }
        if (kWide) *reinterpret_cast<f32x4 *>(&wideStage[l32 * kOutStride + 4 * hl + 32 * nb + 8 * g]) = wide;
        else *reinterpret_cast<v4 *>(pieces + 32 * nb + 8 * g) = o;
      }
#pragma unroll
    for (int it = 0; it < kStoreChunks / 2; it++) {
      const int row = it / kStoreCols * kStoreRowStep;
      u32x4 v;
      if (kWide) {
        v = *reinterpret_cast<const u32x4 *>(&wideStage[row * kOutStride + sat[it % kStoreCols]]);
      } else {
        const uint16_t *p = &stage[(32 * mb + row) * kOutStride + sat[it % kStoreCols]];
        const u32x2 lo = *reinterpret_cast<const u32x2 *>(p);
        const u32x2 hi = *reinterpret_cast<const u32x2 *>(p + 4);
        v = u32x4{lo[0], lo[1], hi[0], hi[1]};
      }
      // (written through to memory; rows that are no whole lines are left to the caches, which put their pieces together: 6000 x 3000
      // x 512 39.7 / 30.8 us, 4096 x 3080 x 160 18 / 13.6)
      if (N % 64) __builtin_amdgcn_raw_buffer_store_b128(v, rows, soff[it % kStoreCols] + (uint32_t)((32 * mb + row) * N * kOutSize), 0, 0);
      else __builtin_amdgcn_raw_buffer_store_b128(v, rows, soff[it % kStoreCols] + (uint32_t)((32 * mb + row) * N * kOutSize), 0, 16);
    }
  }
}

template <typename T, int BN, bool RAGGED>
void launch(const uint16_t *a, const uint16_t *w, const uint16_t *b, const uint16_t *r, uint16_t *o, int64_t M, int64_t N, int64_t K,
            int act, hipStream_t stream) {
  const int tilesM = (int)((M + kBM - 1) / kBM), tilesN = (int)((N + BN - 1) / BN);
  const dim3 grid((unsigned)(tilesM * tilesN)), block(kThreads);
  if (r) launchKernel(gemm_wide_kernel<T, kResidual, BN, uint16_t, RAGGED>, grid, block, stream, a, w, b, r, o, (int)N, (int)K, tilesN, tilesM, (int)M);
  else if (act == ACT_GELU) launchKernel(gemm_wide_kernel<T, ACT_GELU, BN, uint16_t, RAGGED>, grid, block, stream, a, w, b, r, o, (int)N, (int)K, tilesN, tilesM, (int)M);
  else if (act == ACT_RELU) launchKernel(gemm_wide_kernel<T, ACT_RELU, BN, uint16_t, RAGGED>, grid, block, stream, a, w, b, r, o, (int)N, (int)K, tilesN, tilesM, (int)M);
  else launchKernel(gemm_wide_kernel<T, ACT_NONE, BN, uint16_t, RAGGED>, grid, block, stream, a, w, b, r, o, (int)N, (int)K, tilesN, tilesM, (int)M);
  MGPU_CHECK_LAUNCH("gemm_wide_kernel");
}

template <int BN>
void launchToF32(const void *a, const void *w, const void *b, const void *r, float *o, int64_t M, int64_t N, int64_t K, hipStream_t stream) {
  const int tilesM = (int)((M + kBM - 1) / kBM), tilesN = (int)((N + BN - 1) / BN);
  launchKernel(gemm_wide_kernel<_Float16, kResidual, BN, float, false>, dim3((unsigned)(tilesM * tilesN)), dim3(kThreads), stream,
      static_cast<const uint16_t *>(a), static_cast<const uint16_t *>(w), static_cast<const uint16_t *>(b), static_cast<const uint16_t *>(r), o,
      (int)N, (int)K, tilesN, tilesM, (int)M);
  MGPU_CHECK_LAUNCH("gemm_wide_kernel");
}

template <typename T>
void launchWidth(const void *in, const void *weight, const void *bias, const void *residual, void *out, int64_t M, int64_t N, int64_t K,
                 int act, int width, hipStream_t stream) {
  const auto *a = static_cast<const uint16_t *>(in), *w = static_cast<const uint16_t *>(weight), *b = static_cast<const uint16_t *>(bias),
             *r = static_cast<const uint16_t *>(residual);
  auto *o = static_cast<uint16_t *>(out);
  auto at = [&](auto ragged) {
    constexpr bool RAGGED = decltype(ragged)::value;
    if (width == 256) launch<T, 256, RAGGED>(a, w, b, r, o, M, N, K, act, stream);
    else if (width == 192) launch<T, 192, RAGGED>(a, w, b, r, o, M, N, K, act, stream);
    else launch<T, 128, RAGGED>(a, w, b, r, o, M, N, K, act, stream);
  };
  if (K % 64) at(std::true_type());
  else at(std::false_type());
}

} // namespace

bool gemmWideSupports(DType dt, const void *in, const void *weight, const void *bias, const void *residual, const void *out, int64_t M,
                      int64_t N, int64_t K) {
  if (dt != DType::F16 && dt != DType::BF16) return false;
  // 32-bit lane offsets inside a buffer, a slice and a part; fewer than 2^23 tiles of 512 threads
  if (M <= 0 || N <= 0 || N % 8 || K <= 64 || K % 8 || K > (1 << 20) || N > (1 << 20)) return false;
  if (K % 64 && K * N >= int64_t(1) << 30) return false; // (a buffer holds the weight)
  if (M > 0x7fffff00 || (M + kBM - 1) / kBM > 0x7fffff / ((N + 127) / 128)) return false;
  if (!aligned16(in) || !aligned16(weight) || !aligned16(out)) return false;
  if (bias && (reinterpret_cast<uintptr_t>(bias) & 7u)) return false;
  return !residual || aligned16(residual);
}

// Fitted to 1100 shapes (100 to 8192 rows, 128 to 4096 deep, aligned and ragged): 5 % rms, 20 % at worst.  A round of the
// CUs costs its start and end and, per step of the reduction, a part however many CUs take part and - the power limit - a part
// in proportion to them; GELU and the residual come on top.  (us; 4096 x 3072 x 768 + GELU 24.6, 4096 x 6144 x 2048 88.5,
// 4096 x 2048 x 2048 + residual 33.5, 4096 x 2304 x 768 19.8; hipBLASLt 37.9, 107, 37.4, 29.3.)
int gemmWideBest(int64_t M, int64_t N, int64_t K, int act, bool hasResidual, double *cost) {
  struct Width {
    int columns;
    double round, step, shared, gelu, residual;
  };
  static const Width widths[3] = {
      {128, 4.0, 7.25e-3, 4.9e-3, 2.7, 1.95}, {192, 5.2, 10.1e-3, 7.2e-3, 4.0, 3.5}, {256, 6.0, 13.8e-3, 8.5e-3, 5.4, 5.4}};
  const int64_t cus = numComputeUnits();
  K = (K + 63) / 64 * 64; // (what is multiplied)
  int best = 0;
  for (const Width &w : widths) {
    const int64_t tiles = (M + kBM - 1) / kBM * ((N + w.columns - 1) / w.columns), rounds = (tiles + cus - 1) / cus;
    const double full = (double)tiles / (double)cus;
    double us = (double)rounds * (w.round + w.step * (double)K + (act == ACT_GELU ? w.gelu : 0.0)) +
                full * (w.shared * (double)K + (hasResidual ? w.residual : 0.0));
    // Cards differ: on some, short products repeated back to back lose up to half of their rate once more than four fifths of the
    // CUs pull tiles as narrow as these (the clock stays up), on others nothing.  The estimate takes a loss between the two, so that
    // fewer, wider tiles win unless they are much slower (us on such a card / on another, tiles of 128 / 192 / 256 columns: 2048 x 4096 x
    // 512 24 / 13.8 / 14.9 and 11.2 / 12.3 / 14.5, hipBLASLt 15 and 13; 4096 x 2048 x 1024 29 / 21.5 / 21.9 and 18.0 / 19.8 / 22.5, 23 and 21;
    // 4096 x 3072 x 768 36 / 28 / 22.4, 26; not 4096 x 2048 x 2048 35.5 / 39.2 / 40.7, 39.7, nor 6144 x 3072 x 768 51 / 38.6 / 42.3, 42, nor 4096 x
    // 1280 x 768, 160 tiles of 128, 11.8 / 14.0 / 16.7, 15.4).
    const bool crowded = tiles * 5 > cus * 4 && (w.columns == 128 || (w.columns == 192 && rounds == 1));
    if (crowded && K >= 192 && K <= 1408 && act != ACT_GELU) us += w.columns == 128 ? 9.0 : 7.0;
    if (!best || us < *cost) {
      best = w.columns;
      *cost = us;
    }
  }
  return best;
}

void gemmWide(DType dt, const void *in, const void *weight, const void *bias, const void *residual, void *out, int64_t M, int64_t N,
              int64_t K, int act, int width, hipStream_t stream) {
  if (!gemmWideSupports(dt, in, weight, bias, residual, out, M, N, K) || (act != ACT_NONE && residual) ||
      (width != 128 && width != 192 && width != 256))
    fail("gemmWide: internal dispatch error");
  if (dt == DType::F16) launchWidth<_Float16>(in, weight, bias, residual, out, M, N, K, act, width, stream);
  else launchWidth<bf16_t>(in, weight, bias, residual, out, M, N, K, act, width, stream);
}

void gemmWideResidualF32(const void *in, const void *weight, const void *bias, const void *residual, float *out, int64_t M, int64_t N, int64_t K,
                         int width, hipStream_t stream) {
  if (!gemmWideSupports(DType::F16, in, weight, bias, residual, out, M, N, K) || !residual || K % 64) fail("gemmWide: internal dispatch error");
  if (width == 256) launchToF32<256>(in, weight, bias, residual, out, M, N, K, stream);
  else if (width == 192) launchToF32<192>(in, weight, bias, residual, out, M, N, K, stream);
  else launchToF32<128>(in, weight, bias, residual, out, M, N, K, stream);
}

} // namespace mgpu
