// The attention kernel for launches that leave the chip idle: a block owns 32 QG queries (QG = 1 or 2) of one (batch,
// head), and its wavefronts split the KEYS.
//
// fmha_kernel.hpp gives a block 128 queries; a request or two with a few heads is then a few dozen blocks on 256
// CUs, each walking all keys in one chain of waits, barriers and softmaxes.  Here there are two or four times as many
// blocks, and the KS = W / QG wavefronts of a query group take tiles of 32 keys ks, ks + KS, ... of their own.  Each streams
// its K and V tiles HBM -> LDS into a ring of its own (no barrier in the loop; at head_dim 64 all keys of S <= 512 are in
// flight at once) and keeps its own reference maximum, row sum and output.  At the end these meet in LDS in fp32:
//   O = sum_w e_w O_w / sum_w e_w l_w,   e_w = exp2((m_w - max m) c).
// MFMA formulation, LDS swizzles and the stale-reference softmax are those of fmha_kernel.hpp; its head comment has the
// reasons.  K and V are read two or four times as often, which at these sizes the L2 serves.
//
// A chain of latencies still bounds it (launch, first tile, softmax of ceil(S / 32 / KS) tiles, merge), so the time
// hardly grows with the number of blocks up to one round of the CUs.  Measured, fp16, one launch after another, the 128-query
// kernel -> this one: (1, 512, 16 heads of 64) 9.1 -> 6.6 us, (1, 2048, 4 of 64) 28.6 -> 11.2, (1, 512, 16 of 128) 13.2 ->
// 9.0, (1, 507, 8 of 256) 28 -> 15, causal (1, 2048, 16 of 128) 45.6 -> 34.2.  W = 4 with two tiles in
// flight in place of W = 8 with one at head_dim 128: (1, 2048, 4 heads) 24.1 against 17.8.
#include "fmha_kernel.hpp"
#include "mgpu_ops_internal.hpp"

namespace mgpu {

namespace {

using namespace fmha_detail;

template <int D> struct SplitGeo {
  using G = Geo<D>;
  static constexpr int W = D == 256 ? 4 : 8;                // wavefronts of a block
  static constexpr int R = D == 64 ? 2 : 1;                 // ring depth of a wavefront, in tiles
  static constexpr int kTileBytes = 32 * G::rowBytes;       // a K or V tile of 32 keys: 4 / 8 / 16 KiB
  static constexpr int LPT = kTileBytes / 1024;             // loads of 1 KiB per tile: 4 / 8 / 16
  static constexpr int kRingBytes = W * R * 2 * kTileBytes; // 128 KiB: a block has a CU to itself
  static constexpr int OS = D + 4;                          // merge row stride in floats
  static constexpr int kMergeBytes = W * 32 * OS * 4 + W * 32 * 8;
  static constexpr int kLdsBytes = kRingBytes > kMergeBytes ? kRingBytes : kMergeBytes;
  static_assert(kLdsBytes <= 160 * 1024, "LDS of a CU");
};

// (PAD, USED: see fmha_kernel.hpp)
template <typename T, int D, int QG, bool CAUSAL, bool PAD, int USED>
__global__ __launch_bounds__(64 * SplitGeo<D>::W, 1) void fmha_split_kernel(const uint16_t *__restrict__ qkv,
                                                                            const int32_t *__restrict__ seqlens,
                                                                            const int32_t *__restrict__ cuSeqlens,
                                                                            uint16_t *__restrict__ out, int S, int H, int nQB,
                                                                            float scale_log2e, int nblk, int dHead) {
  using M = Mma<T>;
  using v8 = typename M::v8;
  using v4 = typename M::v4;
  using G = Geo<D>;
  using SG = SplitGeo<D>;
  constexpr int DC = (USED + 15) / 16, DB = (USED + 31) / 32, KF = DC < G::KF ? DC : G::KF, VF = DB < G::VF ? DB : G::VF;
  constexpr int W = SG::W, KS = W / QG, R = SG::R, LPT = SG::LPT, kTileBytes = SG::kTileBytes;
  const int kD = PAD ? dHead : D;
  const int validChunks = PAD ? dHead / 8 : G::CPR;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[SG::kLdsBytes];

  // Blocks of one (batch, head) share an XCD's L2 (see fmha_kernel.hpp); under the causal mask its longest block first.
  const int bid = blockIdx.x;
  const int wid = (nblk % 8 == 0) ? (bid % 8) * (nblk / 8) + bid / 8 : bid;
  const int bh = wid / nQB;
  const int item = CAUSAL ? nQB - 1 - wid % nQB : wid % nQB;
  const int h = bh % H, b = bh / H;
  const int tid = threadIdx.x, lane = tid % 64, l32 = lane % 32, hl = lane / 32;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int ks = wave % KS; // this wavefront's share of the keys; its queries are those of group wave / KS

  int kvlen = S, rows = S; // admissible keys; token rows that exist
  size_t tok0 = (size_t)b * S;
  if (cuSeqlens) {
    const int first = cuSeqlens[b];
    kvlen = cuSeqlens[b + 1] - first;
    kvlen = kvlen < 0 ? 0 : (kvlen > S ? S : kvlen);
    rows = kvlen;
    tok0 = (size_t)first;
    if (item * 32 * QG >= rows) return;
  } else if (seqlens) {
    kvlen = seqlens[b];
    kvlen = kvlen < 0 ? 0 : (kvlen > S ? S : kvlen);
  }
  const uint32_t tokBytes = (uint32_t)3 * H * kD * 2;
  const char *qbase = reinterpret_cast<const char *>(qkv) + (tok0 * 3 * H + h) * kD * 2;
  const char *kbase = qbase + (size_t)H * kD * 2;
  const char *vbase = qbase + (size_t)2 * H * kD * 2;
  const int q0 = item * 32 * QG + wave / KS * 32; // first query of this wavefront
  int kend = kvlen;
  if (CAUSAL) kend = kend < q0 + 32 ? kend : q0 + 32;
  // Tiles of 32 keys; this wavefront's are ks, ks + KS, ...  A tile that exists has its first key visible to every
  // query of the wavefront (tiles end with the diagonal one), so its first tile always gives a row a sum.
  const int tiles = q0 < rows ? (kend + 31) / 32 : 0;
  const int n = tiles > ks ? (tiles - ks + KS - 1) / KS : 0;

  // Q as the B operand: lane (query l32, k-slots = d 16c + 8hl .. +7).
  v8 qf[DC];
  {
    int row = q0 + l32;
    row = row < rows ? row : rows - 1;
#pragma unroll
    for (int c = 0; c < DC; c++) {
      if (!PAD || 2 * c + hl < validChunks)
        qf[c] = *reinterpret_cast<const v8 *>(qbase + (size_t)row * tokBytes + (16 * c + 8 * hl) * 2);
      else
        qf[c] = v8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }

  // ---- tile movers: one instruction fills RPI rows; lane l lands in chunk l % CPR of row l / CPR -------------
  const int mrow = lane / G::CPR, mchunk = lane % G::CPR;
  auto srcChunk = [&](int chunk) { return (PAD && chunk >= validChunks) ? 0 : chunk; };
  const uint32_t ldsBase = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) unsigned char *)smem) + (uint32_t)(wave * R * 2 * kTileBytes);
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  auto dma16 = [&](uint32_t voffset, const char *sbase, uint32_t ldsAddr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(voffset), "s"(sbase), "s"(ldsAddr)
                 : "memory", "m0");
  };
#pragma clang diagnostic pop
  auto issueHalf = [&](int j, bool isV) { // K or V of this wavefront's tile j
    const int key0 = (ks + j * KS) * 32;
    const uint32_t dst = ldsBase + (uint32_t)((j % R) * 2 * kTileBytes + (isV ? kTileBytes : 0));
    const char *base = isV ? vbase : kbase;
    const int last = rows - 1 - key0; // (a row beyond the sequence fetches the last one: the mask hides it)
#pragma unroll
    for (int i = 0; i < LPT; i++) {
      const int row = G::RPI * i + mrow;
      const int from = row < last ? row : last;
      dma16((uint32_t)from * tokBytes + (uint32_t)(srcChunk(mchunk ^ (isV ? G::vSwz(row) : G::kSwz(row))) * 16),
            base + (size_t)key0 * tokBytes, dst + i * 1024);
    }
  };
#pragma unroll
  for (int j = 0; j < R; j++)
    if (j < n) {
      issueHalf(j, false);
      issueHalf(j, true);
    }

  // ---- operand addresses inside a tile, as in fmha_kernel.hpp ---------------------------------------------
  uint32_t kfrag[KF], vfrag[VF];
#pragma unroll
  for (int c = 0; c < KF; c++) kfrag[c] = (uint32_t)(l32 * G::rowBytes + (((2 * c + hl) ^ G::kSwz(l32)) * 16));
#pragma unroll
  for (int db = 0; db < VF; db++) {
    const int g = lane / 16, L = lane % 16, r = L % 4, j = L / 4;
    const int chunk = (4 * db + 2 * (g % 2) + r / 2) ^ G::vSwz(4 * hl + j);
    vfrag[db] = (uint32_t)((4 * hl + j) * G::rowBytes + chunk * 16 + 8 * (r % 2));
  }

  f32x16 accO[DB];
  float m_run = 0.0f, l_run = 0.0f; // reference maximum (raw score units), this lane's share of the row sum
#pragma unroll
  for (int db = 0; db < DB; db++)
#pragma unroll
    for (int i = 0; i < 16; i++) accO[db][i] = 0.0f;
  // (a use of every Q register here keeps the wait for them out of the loop)
#pragma unroll
  for (int c = 0; c < DC; c++) asm volatile("" ::"v"(qf[c]));

  // The loads are counted by hand.  In flight, in order: K j, V j, K j+1, V j+1, ... up to tile j+R-1; the K of tile j+R
  // follows the scores of tile j, its V the product with V of tile j.
  for (int j = 0; j < n; j++) {
    const int key0 = (ks + j * KS) * 32;
    const uint32_t stage = ldsBase + (uint32_t)((j % R) * 2 * kTileBytes);
    if (R == 2 && j + 1 < n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * LPT) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPT) : "memory");

    // ---- S^T = K Q^T
    f32x16 accS;
#pragma unroll
    for (int i = 0; i < 16; i++) accS[i] = 0.0f;
#pragma unroll
    for (int c = 0; c < DC; c++) {
      const lds_u8 *kp = (const lds_u8 *)(uintptr_t)(stage + kfrag[c % KF]);
      const v8 a = *reinterpret_cast<const v8 __attribute__((address_space(3))) *>(kp + (c / KF) * 256);
      accS = M::run(a, qf[c], accS);
    }
    const bool more = j + R < n;
    if (more) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the K operands are in registers
      issueHalf(j + R, false);
    }

    if (key0 + 32 > kvlen || (CAUSAL && key0 + 31 > q0)) {
      const int query = q0 + l32;
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int key = key0 + 8 * (i / 4) + 4 * hl + (i % 4);
        if (!(key < kvlen && (!CAUSAL || key <= query))) accS[i] = -INFINITY;
      }
    }
    // ---- P against the stale reference maximum
    v8 pf[2];
    auto makeP = [&](float mref) {
      const float mc = mref * scale_log2e;
      float lsum = 0.0f, lsumOdd = 0.0f;
#pragma unroll
      for (int m = 0; m < 2; m++)
#pragma unroll
        for (int i = 0; i < 8; i++) {
          const float e = __builtin_amdgcn_exp2f(accS[8 * m + i] * scale_log2e - mc);
          (i & 1 ? lsumOdd : lsum) += e;
          pf[m][i] = M::narrow(e);
        }
      return lsum + lsumOdd;
    };
    float lsum = makeP(m_run);
    if (__builtin_amdgcn_ballot_w64(!(lsum <= kSumLimit) || (j == 0 && !(lsum >= kSumFloor))) != 0) {
      float mx = accS[0];
#pragma unroll
      for (int i = 0; i < 16; i++) mx = fmaxf(mx, accS[i]);
      mx = halves_max(mx);
      float m_new, alpha;
      if (j > 0) { // the row has a history: the reference only rises
        m_new = fmaxf(m_run, mx);
        alpha = __builtin_amdgcn_exp2f((m_run - m_new) * scale_log2e);
      } else { // first tile: start over from its maximum
        m_new = mx == -INFINITY ? m_run : mx;
        alpha = 0.0f;
      }
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) accO[db][i] *= alpha;
      lsum = makeP(m_new);
    }
    l_run += lsum;

    // ---- O^T += V^T P^T
    if (R == 2 && j + 1 < n) {
      if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * LPT) : "memory");
      else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LPT) : "memory");
    } else if (R == 1 && more) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPT) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    // Rows of masked keys meet p = 0; zero them so that stray NaN/Inf bits in padding cannot reach the accumulators.
    if (key0 + 32 > kvlen) {
      const lds_u8 *vst = (const lds_u8 *)(uintptr_t)(stage + kTileBytes);
#pragma unroll
      for (int i = 0; i < LPT; i++)
        if (key0 + G::RPI * i + mrow >= kvlen)
          *(u32x4 __attribute__((address_space(3))) *)(vst + i * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
      for (int m = 0; m < 2; m++) {
        const lds_u8 *p = (const lds_u8 *)(uintptr_t)(stage + kTileBytes + vfrag[db % VF]) + (db / VF) * 256 + 16 * m * G::rowBytes;
        const v4 lo = M::readTr(p);
        const v4 hi = M::readTr(p + 8 * G::rowBytes);
        accO[db] = M::run(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), pf[m], accO[db]);
      }
    if (more) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the V operands are in registers
      issueHalf(j + R, true);
    }
  }

  // ---- the shares meet in LDS ---------------------------------------------------------------------------------
  __syncthreads(); // every wavefront is done with its ring
  float *part = reinterpret_cast<float *>(smem); // [W][32][OS]
  float *ml = part + W * 32 * SG::OS;            // [W][32] pairs (reference, row sum)
#pragma unroll
  for (int db = 0; db < DB; db++)
#pragma unroll
    for (int g = 0; g < 4; g++)
      *reinterpret_cast<f32x4 *>(&part[(wave * 32 + l32) * SG::OS + 32 * db + 8 * g + 4 * hl]) =
          f32x4{accO[db][4 * g], accO[db][4 * g + 1], accO[db][4 * g + 2], accO[db][4 * g + 3]};
  const float lAll = halves_sum(l_run);
  if (hl == 0) {
    ml[(wave * 32 + l32) * 2] = m_run;
    ml[(wave * 32 + l32) * 2 + 1] = lAll;
  }
  __syncthreads();
#pragma unroll
  for (int first = 0; first < QG * 32 * G::CPR; first += 64 * W) {
    const int chunk = first + tid; // 16-byte chunk of the output tile
    if (chunk >= QG * 32 * G::CPR) break;
    const int r = chunk / G::CPR, cidx = chunk % G::CPR;
    const int query = item * 32 * QG + r;
    const int row0 = r / 32 * KS * 32 + r % 32; // the row in the share of the group's first wavefront
    if (query >= rows || (PAD && cidx >= validChunks)) continue;
    float top = -INFINITY;
#pragma unroll
    for (int w = 0; w < KS; w++) // (a wavefront without a tile has a row sum of 0 and no say)
      if (ml[(w * 32 + row0) * 2 + 1] != 0.0f) top = fmaxf(top, ml[(w * 32 + row0) * 2]);
    float l = 0.0f, o[8] = {};
#pragma unroll
    for (int w = 0; w < KS; w++) {
      const float lw = ml[(w * 32 + row0) * 2 + 1];
      const float e = lw != 0.0f ? __builtin_amdgcn_exp2f((ml[(w * 32 + row0) * 2] - top) * scale_log2e) : 0.0f;
      l += e * lw;
      const float *src = &part[(w * 32 + row0) * SG::OS + cidx * 8];
      const f32x4 lo = *reinterpret_cast<const f32x4 *>(src), hi = *reinterpret_cast<const f32x4 *>(src + 4);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        o[i] += e * lo[i];
        o[4 + i] += e * hi[i];
      }
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    v8 val;
#pragma unroll
    for (int i = 0; i < 8; i++) val[i] = M::narrow(o[i] * inv);
    *reinterpret_cast<v8 *>(out + (tok0 + query) * H * kD + (size_t)h * kD + cidx * 8) = val;
  }
}

// Query groups of a block, 0 where the 128-query kernel is as fast or faster.  D is the tile geometry.
//  * One group while a block per CU covers the launch, two while blocks of 64 queries do: beyond, rounds of blocks that
//    each have a CU to themselves lose to the other kernel's two or three blocks per CU ((1, 512, 64 heads of 64)
//    9.7 us against 14.7; four groups of two key shares at 10.4-11.1 never won by more than 5 %).
//  * Sequences long enough to be worth the merge.  Lengths at which a side is ahead, 128-query kernel / one group / two
//    groups in us - head_dim 64: S = 160 5.3 / 5.1 / 5.6, 192 5.0 / 5.2 / 5.8, 193 6.1 / 5.7 / 6.2, 256 5.8 / 5.4 / 5.9, 257 6.9 /
//    6.0 / 6.9, 320 6.6 / 5.8 / 6.8, 321 7.7 / 6.0 / 6.9, 384 7.4 / 5.9 / 6.7 (one group from 193 on; two are now ahead, now behind by
//    2 % up to 320, from 321 on ahead by 5 % and more); 128: S = 128 5.9 /
//    6.1 / 7.4, 192 7.2 / 7.0 / 8.6, 256 8.5 / 7.5 / 8.9, 384 10.8 / 7.9 / 9.9; 256: S = 64 7.1 / 8.2, 96 9.0 / 8.9 / 11.3,
//    192 13.8 / 11.0 / 13.7, 256 16.8 / 11.6 / 15.6.  The causal mask leaves the 128-query blocks unequal: head_dim 64
//    S = 64 4.1 / 4.8, 96 5.9 / 5.1 / 4.9; 128: S = 64 5.3 / 5.6, 96 7.5 / 6.4 / 6.8, 192 7.7 / 7.4 / 8.6, 256 9.7 / 7.7 / 8.8.
//  * Long causal launches of up to two rounds: 128-query blocks of up to 16 different lengths, one per CU, run as
//    long as the longest ((1, 2048, 16 heads) at head_dim 64 / 128 / 256: 33.4 / 45.6 / 102 us against 22.9 / 34.2 / 77;
//    S = 1024, 32 heads: 18.4 / 24.8 / 54 against 18.7 / 27.7 / 63; three rounds lose at S = 2048 as well).
int splitGroups(int D, int B, int S, int H, bool causal) {
  const int64_t cus = numComputeUnits(), bh = (int64_t)B * H;
  const int from1 = D == 256 || causal ? 65 : D == 128 ? 129 : 193; // shortest sequences for one group
  const int from2 = D == 64 ? (causal ? 65 : 321) : D == 128 && !causal ? 257 : 193; // and for two
  if (bh * ((S + 31) / 32) <= cus) return S >= from1 ? 1 : 0;
  const int64_t blocks2 = bh * ((S + 63) / 64);
  if (blocks2 <= cus) return S >= from2 ? 2 : 0;
  return causal && S >= 2048 && blocks2 <= 2 * cus ? 2 : 0;
}

template <typename T, int D, int QG, bool PAD, int USED = D>
void launchSplit(const void *qkv, const int32_t *seqlens, const int32_t *cuSeqlens, void *out, int B, int S, int H,
                 int dHead, float scale, bool causal, hipStream_t stream) {
  const int nQB = (S + 32 * QG - 1) / (32 * QG);
  const unsigned blocks = (unsigned)B * H * nQB; // at most two per CU
  const float c = scale * 1.44269504088896340736f;
  const auto *in = static_cast<const uint16_t *>(qkv);
  auto *o = static_cast<uint16_t *>(out);
  const dim3 grid(blocks), block(64 * SplitGeo<D>::W);
  if (causal)
    launchKernel(fmha_split_kernel<T, D, QG, true, PAD, USED>, grid, block, stream, in, seqlens, cuSeqlens, o, S, H, nQB, c, (int)blocks, dHead);
  else
    launchKernel(fmha_split_kernel<T, D, QG, false, PAD, USED>, grid, block, stream, in, seqlens, cuSeqlens, o, S, H, nQB, c, (int)blocks, dHead);
  MGPU_CHECK_LAUNCH("fmha_split_kernel");
}

template <typename T, int D>
bool launchGeometry(const void *qkv, const int32_t *seqlens, const int32_t *cuSeqlens, void *out, int B, int S, int H,
                    int dHead, float scale, bool causal, hipStream_t stream) {
  const int groups = splitGroups(D, B, S, H, causal);
  if (groups == 0) return false;
  constexpr int kFew = D == 64 ? 32 : D == 128 ? 80 : 160, kSome = D == 64 ? 48 : D == 128 ? 96 : 160; // (as in fmha.hip)
  auto pick = [&](auto qg) {
    constexpr int QG = decltype(qg)::value;
    return dHead == D ? launchSplit<T, D, QG, false> : dHead <= kFew ? launchSplit<T, D, QG, true, kFew>
           : dHead <= kSome ? launchSplit<T, D, QG, true, kSome> : launchSplit<T, D, QG, true>;
  };
  const auto launch = groups == 1 ? pick(std::integral_constant<int, 1>()) : pick(std::integral_constant<int, 2>());
  launch(qkv, seqlens, cuSeqlens, out, B, S, H, dHead, scale, causal, stream);
  return true;
}

} // namespace

bool fusedMHASplitKeys(DType dt, const void *qkv, const int32_t *seqlens, const int32_t *cuSeqlens, void *out, int B, int S,
                       int H, int D, float scale, bool causal, hipStream_t stream) {
  auto go = [&](auto type) {
    using T = decltype(type);
    const auto launch = D <= 64 ? launchGeometry<T, 64> : D <= 128 ? launchGeometry<T, 128> : launchGeometry<T, 256>;
    return launch(qkv, seqlens, cuSeqlens, out, B, S, H, D, scale, causal, stream);
  };
  return dt == DType::F16 ? go(_Float16{}) : go(bf16_t{});
}

} // namespace mgpu
