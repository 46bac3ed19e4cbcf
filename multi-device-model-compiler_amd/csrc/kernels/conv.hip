// 2-D convolution and pooling on NCHW fp32 tensors.
//
// Replaces mgpuConv2d and mgpuPool2d (lib/Kernels/GPU/Ops.cu:238-335,337-374;
// declared in Ops.h:27-41), which wrap cudnnConvolutionBiasActivationForward and
// cudnnPoolingForward:
//   conv:  y = act(conv(x, w) + bias[oc] + postAdd),  act = ReLU or identity
//   pool:  max (padding ignored) or average that counts the padding
//          (CUDNN_POOLING_AVERAGE_COUNT_INCLUDE_PADDING, Ops.cu:347-349)
// The convolution is an implicit GEMM, mostly on the fp32 matrix cores
// (v_mfma_f32_32x32x2_f32: true fp32 products, fp32 accumulation):
//   y[n][oc, p] = sum_k w[oc, k] * taps[k, p],  k = (ic, kh, kw), p = (oh, ow)
// in 32 x 32 tiles, channels in the rows and pixels - counted over the whole batch - in the
// columns, so that a register of an accumulator is 32 consecutive pixels of a channel: whole
// 128-byte runs of the NCHW output.  The tap matrix is never written to memory.  Taps come
// through buffer loads, whose bounds check answers 0 for an offset outside the image: padding costs
// no branch and no second instruction.  Seven kernels share the work here (conv2d below has the rule and
// the measurements behind it), with two more: conv_small.hip takes 3 x 3, 5 x 5 and 7 x 7 of few tiles, in tiles of 16 pixels, and
// conv_split.hip the large ones, on the bf16 matrix cores in three numbers an operand, as the quads of 12 taps on are here:
//   few taps  (K <= 32, a network's stem)  filter in registers, wavefronts walk over pixel tiles
//   quads     (the same, many tiles, rows of whole quads, stride 1 across)  four pixels a lane
//   patch     (5 or 7 square from one channel or three)  input rows through LDS, once for all taps
//   window    (1, 3, 5 or 7 square, few tiles)  operands straight from L1 / L2 into registers,
//             four wavefronts per tile
//   staged    (3, 5 or 7 square, even channels, few tiles)  the same with the filter through LDS
//   tile      (the same windows, many tiles)    operands shared through LDS by 64 x 64 tiles
//   table     (every other window, and images beyond 2 GiB)  tap offsets from a table in LDS
// What bounds them: one 32x32x2 MFMA takes 64 cycles of a SIMD (157 TFLOP/s on the chip) and the
// vector instructions of the same wavefront do not overlap with it, so the loops are built to have
// none; the stem is bound by its output (268 MB at 16 x 3 x 256 x 256 -> 64: 55 us, a plain fill
// of as many bytes takes 39).  Unlike the reference, asymmetric padding is honoured (it passes only
// PHL / PWL to cuDNN).
#include "common.hpp"
#include "conv.hpp"
#include "mgpu_ops_internal.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace mgpu {

namespace {

struct ConvGeo {
  int IC, H, W, KH, KW, OH, OW, PHL, PWL, SH, SW, DH, DW;
};

constexpr int kChunk = 16;     // taps per step of the reduction: 8 a lane half
constexpr int kSegment = 2048; // taps the tap table holds at a time
constexpr int kNever = 0x3fff0000; // a pixel past the end takes -kNever for its first row: every tap lies outside the image

// Where tap k of a pixel sits: the offset from the pixel's first tap (bytes; elements when WIDE)
// and the window position (kw | kh << 5) or, for WIDE (images beyond 2 GiB, windows beyond 31
// positions), the row and column distances.
struct TapNarrow {
  int off, pos;
};
struct TapWide {
  int off, dh, dw, pad;
};

// Which of `count` window rows (columns), `dilation` apart from `first` on, lie outside 0 .. size - 1: bit i for the i-th.
__device__ __forceinline__ unsigned outsideBits(int first, int size, int count, int dilation) {
  if (dilation == 1) { // (uniform) the bits below -first and from size - first on
    const int lo = first < 0 ? -first : 0, hi = size - first;
    const unsigned below = lo > 31 ? ~0u : (1u << lo) - 1u, above = hi > 31 ? 0u : hi < 0 ? ~0u : ~0u << hi;
    return below | above;
  }
  unsigned bits = 0;
  for (int i = 0; i < count; i++) bits |= (unsigned)(first + i * dilation) < (unsigned)size ? 0u : 1u << i;
  return bits;
}

// A launch holds fewer than 2^32 threads in one dimension: beyond, the row of pixel blocks goes on in blockIdx.z, 2^31
// threads at a time (gridOf in conv2d), and the last piece has blocks past the last pixel.
constexpr int64_t kGridRow = int64_t(1) << 31;
template <int THREADS> __device__ __forceinline__ int pixelBlock() { return (int)blockIdx.z * (int)(kGridRow / THREADS) + (int)blockIdx.x; }

// The end of a wavefront's 32 channels x PT x 32 pixels: the sum over the KS wavefronts of the tile
// (wavefront ks of them has slot `slot0` + ks of `partial`), bias, postAdd, ReLU, store.  pix and img:
// the lane's pixels (-1: past the end) and their images less nFirst.  Lane: the type of a lane's byte
// offset from image nFirst.
template <int PT, int KS, typename Lane, int SLOTS, int WORDS>
__device__ __forceinline__ void finishTile(f32x16 (&acc)[PT], float (&partial)[SLOTS][WORDS], int slot0, int ks, const float *bias,
                                           const float *add, float *y, int OC, int P, int oc0, int nFirst, const int (&img)[PT],
                                           const int (&pix)[PT], int lane, int relu) {
  const int hl = lane / 32;
  // accumulator register r of lane l: channel 8*(r/4) + 4*(l/32) + r%4, pixel l%32.  (Offsets are
  // bytes next to a uniform base: a store takes its address from a scalar pair and one vector register.)
  const int64_t first = ((int64_t)nFirst * OC + oc0) * P;
  Lane at[PT];
#pragma unroll
  for (int j = 0; j < PT; j++) at[j] = (((Lane)img[j] * OC + 4 * hl) * P + (Lane)pix[j]) * 4;
  constexpr int SHARE = 16 / KS; // registers this wavefront finishes
  if constexpr (KS > 1) {
    static_assert(PT == 1, "one accumulator per wavefront where the taps are split");
#pragma unroll
    for (int r = 0; r < 16; r++) partial[slot0 + ks][r * 64 + lane] = acc[0][r];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < SHARE; i++) {
      float v = 0.0f;
#pragma unroll
      for (int s = 0; s < KS; s++) v += partial[slot0 + s][(ks * SHARE + i) * 64 + lane];
      acc[0][i] = v;
    }
  }
  const bool fullOc = oc0 + 32 <= OC; // (uniform: no channel test inside a full tile)
  auto channel = [&](int i) { // of register i of the wavefront's share, less the lane's 4 hl
    const int r = ks * SHARE + i;
    return 8 * (r / 4) + r % 4;
  };
  float bv[SHARE];
#pragma unroll
  for (int i = 0; i < SHARE; i++) {
    const int oc = oc0 + channel(i) + 4 * hl;
    bv[i] = bias[fullOc || oc < OC ? oc : OC - 1];
  }
  auto epilogue = [&](auto everyChannel, auto plain) {
#pragma unroll
    for (int j = 0; j < PT; j++) {
      if (pix[j] < 0) continue;
#pragma unroll
      for (int i = 0; i < SHARE; i++) {
        const int ocl = channel(i);
        if (!decltype(everyChannel)::value && oc0 + ocl + 4 * hl >= OC) continue;
        const int64_t row = first + (int64_t)ocl * P;
        float v = acc[j][i] + bv[i];
        if (!decltype(plain)::value) v += *reinterpret_cast<const float *>(reinterpret_cast<const char *>(add + row) + at[j]);
        // cuDNN's ReLU with CUDNN_NOT_PROPAGATE_NAN maps NaN to 0, as fmaxf does
        *reinterpret_cast<float *>(reinterpret_cast<char *>(y + row) + at[j]) = relu ? fmaxf(v, 0.0f) : v;
      }
    }
  };
  if (!add && fullOc) epilogue(std::true_type(), std::true_type());
  else if (!add) epilogue(std::false_type(), std::true_type());
  else if (fullOc) epilogue(std::true_type(), std::false_type());
  else epilogue(std::false_type(), std::false_type());
}

// ---- any window -----------------------------------------------------------------------------
// The four wavefronts of a block share one 32 x 32 tile and split the taps.
template <bool WIDE>
__global__ __launch_bounds__(256, 2) void conv_table_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                            const float *__restrict__ bias, const float *__restrict__ add,
                                                            float *__restrict__ y, ConvGeo g, int OC, int K, int P, int64_t pixelsArg,
                                                            int relu) {
  using Tap = typename std::conditional<WIDE, TapWide, TapNarrow>::type;
  using Index = typename std::conditional<WIDE, int64_t, int>::type; // (64-bit divisions are long sequences)
  const Index pixels = (Index)pixelsArg;
  constexpr int KS = 4;
  __shared__ __attribute__((aligned(16))) Tap table[kSegment];
  __shared__ float partial[KS][16 * 64];

  const int tid = threadIdx.x, lane = tid % 64;
  const int ks = __builtin_amdgcn_readfirstlane(tid / 64);
  const int l32 = lane % 32, hl = lane / 32;
  const int oc0 = blockIdx.y * 32;
  const Index q0 = (Index)pixelBlock<256>() * 32;
  if (q0 >= pixels) return;
  const int64_t imageElems = (int64_t)g.IC * g.H * g.W;

  // The lane's pixel.  Which window rows and columns fall outside the image is a bit mask (bit 31
  // always set: the position of a tap past the end); a pixel past the end has every bit set.
  const int nFirst = __builtin_amdgcn_readfirstlane((int)(q0 / P));
  const Index q = q0 + l32;
  const bool live = q < pixels;
  const int n = live ? (int)(q / P) : nFirst;
  const int p = live ? (int)(q - (Index)n * P) : 0;
  const int oh = p / g.OW, ow = p - oh * g.OW;
  const int img[1] = {n - nFirst}, pix[1] = {live ? p : -1};
  const int ih0 = oh * g.SH - g.PHL, iw0 = ow * g.SW - g.PWL;
  Index base = (Index)img[0] * (Index)imageElems + (Index)(oh * g.SH - g.PHL) * g.W + iw0;
  const float *image = x + nFirst * imageElems;
  unsigned rowOut = 0, colOut = 0;
  if constexpr (!WIDE) {
    rowOut = live ? outsideBits(ih0, g.H, g.KH, g.DH) : ~0u;
    colOut = outsideBits(iw0, g.W, g.KW, g.DW) | 0x80000000u;
    base *= 4; // bytes from `image`, in the 32 bits that the host has checked they fit
  }
  const auto rsrc = resource(image, ((pixels - 1) / P + 1 - nFirst) * imageElems);
  const float *wrow = w + (int64_t)(oc0 + l32 < OC ? oc0 + l32 : OC - 1) * K; // (a channel past the end is not stored)

  f32x16 acc[1];
#pragma unroll
  for (int i = 0; i < 16; i++) acc[0][i] = 0.0f;

  // One step's operands: the contraction does not care in which slot a tap sits, so lane half hl
  // takes taps 8 hl .. 8 hl + 7 of the chunk (two 16-byte filter loads) and MFMA i of the step
  // multiplies tap i of either half.
  struct Operands {
    float a[8], b[8];
  };
  auto fetch = [&](Operands &o, int seg, int k) { // taps k .. k + 15, k relative to the segment
    const int kl = k + 8 * hl;
    if (seg + k + kChunk <= K) { // (uniform)
      const f32x4 lo = *reinterpret_cast<const f32x4 __attribute__((aligned(4))) *>(wrow + seg + kl);
      const f32x4 hi = *reinterpret_cast<const f32x4 __attribute__((aligned(4))) *>(wrow + seg + kl + 4);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        o.a[i] = lo[i];
        o.a[4 + i] = hi[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const bool in = seg + kl + i < K;
        const float v = wrow[in ? seg + kl + i : 0];
        o.a[i] = in ? v : 0.0f;
      }
    }
    if constexpr (WIDE) {
#pragma unroll
      for (int i = 0; i < 8; i++) {
        // (pixels and taps past the end are ruled out by their index: a sentinel row for either could meet the other's)
        const Tap tap = table[kl + i];
        const bool in = live && (seg + k + kChunk <= K || seg + kl + i < K) && (unsigned)(ih0 + tap.dh) < (unsigned)g.H &&
                        (unsigned)(iw0 + tap.dw) < (unsigned)g.W;
        const float v = image[in ? base + tap.off : 0];
        o.b[i] = in ? v : 0.0f;
      }
    } else {
      i32x4 e[4]; // two taps each
#pragma unroll
      for (int i = 0; i < 4; i++) e[i] = reinterpret_cast<const i32x4 *>(&table[kl])[i];
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int off = e[i / 2][2 * (i % 2)], pos = e[i / 2][2 * (i % 2) + 1];
        // all ones where the row or the column is outside: two bit-field extracts, an add and an or
        const int out = __builtin_amdgcn_sbfe(rowOut, pos >> 5, 1) | __builtin_amdgcn_sbfe(colOut, pos, 1);
        o.b[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, ((int)base + off) | out, 0, 0));
      }
    }
  };
  auto multiply = [&](const Operands &o) {
#pragma unroll
    for (int i = 0; i < 8; i++) acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(o.a[i], o.b[i], acc[0], 0, 0, 0);
  };

  for (int seg = 0; seg < K; seg += kSegment) {
    const int taps = K - seg < kSegment ? K - seg : kSegment;
    const int padded = (taps + kChunk - 1) / kChunk * kChunk;
    if (seg) __syncthreads(); // everybody is done with the previous segment's table
    for (int e = tid; e < padded; e += 256) {
      const int k = seg + e;
      const int ic = k / (g.KW * g.KH), r = k - ic * (g.KW * g.KH);
      const int kh = r / g.KW, kw = r - kh * g.KW;
      Tap tap;
      tap.off = (ic * g.H + kh * g.DH) * g.W + kw * g.DW;
      if constexpr (WIDE) {
        tap.dh = kh * g.DH;
        tap.dw = kw * g.DW;
        tap.pad = 0;
      } else {
        tap.off = k < K ? tap.off * 4 : 0;
        tap.pos = k < K ? kw | kh << 5 : 31;
      }
      table[e] = tap;
    }
    __syncthreads();

    const int chunks = padded / kChunk;
    const int c0 = chunks * ks / KS, c1 = chunks * (ks + 1) / KS; // this wavefront's share
    // each chunk's loads fly under the MFMAs of the one before
    Operands even, odd;
    if (c0 < c1) fetch(even, seg, c0 * kChunk);
    for (int c = c0; c < c1; c += 2) {
      if (c + 1 < c1) fetch(odd, seg, (c + 1) * kChunk);
      multiply(even);
      if (c + 1 >= c1) break;
      if (c + 2 < c1) fetch(even, seg, (c + 2) * kChunk);
      multiply(odd);
    }
  }

  using Lane = typename std::conditional<WIDE, int64_t, uint32_t>::type;
  finishTile<1, KS, Lane>(acc, partial, 0, ks, bias, add, y, OC, P, oc0, nFirst, img, pix, lane, relu);
}

// ---- square windows of 1, 3, 5 or 7 --------------------------------------------------------
// No tap table: the reduction walks input channels in groups - pairs, one channel per lane half;
// 1 x 1: sixteen, eight per half - and inside a group the window positions, with a register each for
// the position's byte offset.  The channel enters through the scalar offset of the load, so a tap
// costs no vector instruction (the table's five a tap were 40 % of a 32 x 32 tile's loop).
template <int WIN> struct Window {
  static constexpr int KK = WIN * WIN;
  static constexpr int UNITS = WIN <= 3 ? 1 : WIN;        // fetched at a time: the window, or one of its rows
  static constexpr int STEPS = WIN == 1 ? 8 : KK / UNITS; // MFMA steps per unit
  static constexpr int HALF = WIN == 1 ? 8 : 1;           // channels per lane half and group
};

// A wavefront's tile is 32 channels x PT x 32 pixels; KS of a block's four wavefronts share a tile
// and split the channel groups.
template <int WIN, int PT, int KS>
__global__ __launch_bounds__(256, 2) void conv_window_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                             const float *__restrict__ bias, float *__restrict__ y, ConvGeo g, int OC,
                                                             int P, int N, FastDiv byP, FastDiv byOW, const float *__restrict__ add,
                                                             int relu) {
  using Win = Window<WIN>;
  constexpr int KK = Win::KK, UNITS = Win::UNITS, STEPS = Win::STEPS, HALF = Win::HALF;
  constexpr int TILES = 4 / KS;
  __shared__ float partial[KS > 1 ? 4 : 1][KS > 1 ? 16 * 64 : 1];

  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int l32 = lane % 32, hl = lane / 32;
  const int ks = wave % KS, tile = wave / KS;
  const int oc0 = blockIdx.y * 32;
  const int q0 = (pixelBlock<256>() * TILES + tile) * (32 * PT);
  const int HW4 = g.H * g.W * 4, pixels = N * P;

  const int nFirst = __builtin_amdgcn_readfirstlane(divide(q0 < pixels ? q0 : pixels - 1, byP));
  int pix[PT], img[PT], voff[PT][KK];
#pragma unroll
  for (int j = 0; j < PT; j++) {
    const int q = q0 + 32 * j + l32;
    const bool live = q < pixels;
    const int n = live ? divide(q, byP) : nFirst;
    const int p = live ? q - n * P : 0;
    const int oh = divide(p, byOW), ow = p - oh * g.OW;
    img[j] = n - nFirst;
    pix[j] = live ? p : -1;
    const int ih0 = live ? oh * g.SH - g.PHL : -kNever, iw0 = ow * g.SW - g.PWL;
    const int base = (img[j] * g.IC + hl * HALF) * HW4 + ((oh * g.SH - g.PHL) * g.W + iw0) * 4;
#pragma unroll
    for (int kh = 0; kh < WIN; kh++)
#pragma unroll
      for (int kw = 0; kw < WIN; kw++) {
        const bool in = (unsigned)(ih0 + kh * g.DH) < (unsigned)g.H && (unsigned)(iw0 + kw * g.DW) < (unsigned)g.W;
        voff[j][kh * WIN + kw] = in ? base + (kh * g.DH * g.W + kw * g.DW) * 4 : kOutside;
      }
  }
  const int64_t imageElems = (int64_t)g.IC * g.H * g.W;
  const auto image = resource(x + nFirst * imageElems, (N - nFirst) * imageElems);
  const auto filter = resource(w + (int64_t)oc0 * g.IC * KK, (int64_t)(OC - oc0) * g.IC * KK);
  // (a channel past the end reads the last one's filter and is not stored)
  const int woff = ((oc0 + l32 < OC ? l32 : OC - 1 - oc0) * g.IC + hl * HALF) * (KK * 4);

  f32x16 acc[PT];
#pragma unroll
  for (int j = 0; j < PT; j++)
#pragma unroll
    for (int i = 0; i < 16; i++) acc[j][i] = 0.0f;

  struct Operands {
    float a[STEPS], b[PT][STEPS];
  };
  auto loadF = [](const __amdgpu_buffer_rsrc_t &r, int voffset, int soffset) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voffset, soffset, 0));
  };
  auto fetch = [&](Operands &o, int group, auto unitConst) { // a group all of whose channels exist
    constexpr int unit = decltype(unitConst)::value;
    constexpr int AT = unit * STEPS * 4;
    const int wbase = group * (2 * HALF * KK * 4);
#pragma unroll
    for (int i = 0; i + 4 <= STEPS; i += 4) {
      const auto v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(filter, woff + AT + i * 4, wbase, 0));
#pragma unroll
      for (int e = 0; e < 4; e++) o.a[i + e] = v[e];
    }
#pragma unroll
    for (int i = STEPS / 4 * 4; i < STEPS; i++) o.a[i] = loadF(filter, woff + AT + i * 4, wbase);
#pragma unroll
    for (int i = 0; i < STEPS; i++)
#pragma unroll
      for (int j = 0; j < PT; j++)
        o.b[j][i] = loadF(image, voff[j][WIN == 1 ? 0 : unit * STEPS + i], (group * (2 * HALF) + (WIN == 1 ? i : 0)) * HW4);
  };
  auto multiply = [&](const Operands &o) {
#pragma unroll
    for (int i = 0; i < STEPS; i++)
#pragma unroll
      for (int j = 0; j < PT; j++) acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(o.a[i], o.b[j][i], acc[j], 0, 0, 0);
  };

  const int groups = g.IC / (2 * HALF);
  const int g0 = groups * ks / KS, g1 = groups * (ks + 1) / KS; // this wavefront's share
  // Two buffers; a unit's loads fly under the MFMAs of the one before.  With an odd number of units
  // a group ends on the other buffer than it began: the loop body is two groups.
  Operands buf[2];
  if (g0 < g1) fetch(buf[0], g0, std::integral_constant<int, 0>());
  auto oneGroup = [&](int group, auto phaseConst) {
    constexpr int phase = decltype(phaseConst)::value;
    auto step = [&](auto self, auto unitConst) {
      constexpr int unit = decltype(unitConst)::value;
      if constexpr (unit < UNITS) {
        if constexpr (unit + 1 < UNITS) fetch(buf[(phase + unit + 1) % 2], group, std::integral_constant<int, unit + 1>());
        else if (group + 1 < g1) fetch(buf[(phase + unit + 1) % 2], group + 1, std::integral_constant<int, 0>());
        multiply(buf[(phase + unit) % 2]);
        self(self, std::integral_constant<int, unit + 1>());
      }
    };
    step(step, std::integral_constant<int, 0>());
  };
  for (int group = g0; group < g1; group += 2) {
    oneGroup(group, std::integral_constant<int, 0>());
    if (group + 1 < g1) oneGroup(group + 1, std::integral_constant<int, UNITS % 2>());
  }
  // The channels beyond the last whole group: what lies past the last channel is asked for at an
  // offset outside the resource (and reads as 0), operand by operand.
  const int rest = g.IC - groups * (2 * HALF);
  if (rest && ks == KS - 1) {
    auto tail = [&](auto self, auto unitConst) {
      constexpr int unit = decltype(unitConst)::value;
      if constexpr (unit < UNITS) {
        const int wbase = groups * (2 * HALF * KK * 4);
#pragma unroll
        for (int i = 0; i < STEPS; i++) {
          const int c = WIN == 1 ? i : 0; // channel of the step inside the lane half's
          const bool in = hl * HALF + c < rest;
          buf[0].a[i] = loadF(filter, in ? woff + (unit * STEPS + i) * 4 + wbase : kOutside, 0);
#pragma unroll
          for (int j = 0; j < PT; j++) {
            const int at = voff[j][WIN == 1 ? 0 : unit * STEPS + i];
            buf[0].b[j][i] = loadF(image, in && at != kOutside ? at + (groups * (2 * HALF) + c) * HW4 : kOutside, 0);
          }
        }
        multiply(buf[0]);
        self(self, std::integral_constant<int, unit + 1>());
      }
    };
    tail(tail, std::integral_constant<int, 0>());
  }
  finishTile<PT, KS, uint32_t>(acc, partial, tile * KS, ks, bias, add, y, OC, P, oc0, nFirst, img, pix, lane, relu);
}

// The same for few tiles, one of 32 x 32 a block: the filter through LDS.  A matrix instruction wants one value of each of 32
// channels, whose rows lie IC * KK floats apart: loaded straight into registers every instruction touches 32 lines, and the CU's
// one L1, not its four SIMDs, set the pace (8 x 256 x 7 x 7 -> 512, 3 x 3: 20.8 us, 14 with the filter loads of all
// channels on one line, 7.7 by the matrix cores; now 16.8).  Here a wavefront loads its channels' rows along the rows - CG channel groups
// at a time, 16 bytes a lane, under the matrix instructions of the groups before -, keeps them in an LDS area of its own (no
// barrier) and reads an operand a step from there.
template <int WIN> struct Staged {
  static constexpr int CG = WIN == 7 ? 1 : WIN == 5 ? 2 : 4;           // channel groups staged at a time
  static constexpr int ROW = CG * 2 * Window<WIN>::HALF * WIN * WIN;   // floats of a channel's row among them
  static constexpr int PIECE = ROW % 4 == 0 ? 4 : 2;                   // floats loaded at a time
  static constexpr int PIECES = ROW / PIECE, LOADS = (32 * PIECES + 63) / 64;
  static constexpr int PITCH = ROW % 16 == 0 ? ROW + 4 : ROW + (ROW % 8 == 0 ? 4 : 0); // 4 or 12 modulo 16 words, or 98 of 7 x 7, 2 times an odd number: 16 rows on different banks
};
template <int WIN, int KS>
__global__ __launch_bounds__(64 * KS, 2) void conv_staged_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                                 const float *__restrict__ bias, float *__restrict__ y, ConvGeo g, int OC,
                                                                 int P, int N, FastDiv byP, FastDiv byOW, const float *__restrict__ add,
                                                                 int relu) {
  using Win = Window<WIN>;
  using St = Staged<WIN>;
  constexpr int KK = Win::KK, UNITS = Win::UNITS, STEPS = Win::STEPS, HALF = Win::HALF;
  constexpr int kRows = 32 * St::PITCH;
  __shared__ __attribute__((aligned(16))) float smem[KS * (kRows > 16 * 64 ? kRows : 16 * 64)];

  const int tid = threadIdx.x, lane = tid % 64;
  const int ks = __builtin_amdgcn_readfirstlane(tid / 64);
  const int l32 = lane % 32, hl = lane / 32;
  const int oc0 = blockIdx.y * 32, q0 = pixelBlock<64 * KS>() * 32;
  const int HW4 = g.H * g.W * 4, pixels = N * P;

  const int nFirst = __builtin_amdgcn_readfirstlane(divide(q0 < pixels ? q0 : pixels - 1, byP));
  // A tap's byte offset, kOutside where it lies outside; 7 x 7, whose 49 would not leave the registers for the filter: the first
  // window row's, and in bit 31 - kh of rowOut which rows lie outside.
  int pix[1], img[1], voff[WIN == 7 ? WIN : KK];
  unsigned rowOut = 0;
  {
    const int q = q0 + l32;
    const bool live = q < pixels;
    const int n = live ? divide(q, byP) : nFirst;
    const int p = live ? q - n * P : 0;
    const int oh = divide(p, byOW), ow = p - oh * g.OW;
    img[0] = n - nFirst;
    pix[0] = live ? p : -1;
    const int ih0 = live ? oh * g.SH - g.PHL : -kNever, iw0 = ow * g.SW - g.PWL;
    const int base = (img[0] * g.IC + hl * HALF) * HW4 + ((oh * g.SH - g.PHL) * g.W + iw0) * 4;
    if constexpr (WIN == 7) {
#pragma unroll
      for (int k = 0; k < WIN; k++) {
        voff[k] = (unsigned)(iw0 + k * g.DW) < (unsigned)g.W ? base + k * g.DW * 4 : kOutside;
        rowOut |= (unsigned)(ih0 + k * g.DH) < (unsigned)g.H ? 0u : 0x80000000u >> k;
      }
    } else {
#pragma unroll
      for (int kh = 0; kh < WIN; kh++)
#pragma unroll
        for (int kw = 0; kw < WIN; kw++) {
          const bool in = (unsigned)(ih0 + kh * g.DH) < (unsigned)g.H && (unsigned)(iw0 + kw * g.DW) < (unsigned)g.W;
          voff[kh * WIN + kw] = in ? base + (kh * g.DH * g.W + kw * g.DW) * 4 : kOutside;
        }
    }
  }
  const int64_t imageElems = (int64_t)g.IC * g.H * g.W;
  const auto image = resource(x + nFirst * imageElems, (N - nFirst) * imageElems);
  const auto filter = resource(w + (int64_t)oc0 * g.IC * KK, (int64_t)(OC - oc0) * g.IC * KK);

  f32x16 acc[1];
#pragma unroll
  for (int i = 0; i < 16; i++) acc[0][i] = 0.0f;

  const int groups = g.IC / (2 * HALF); // (whole: the launcher sees to it)
  const int g0 = groups * ks / KS, g1 = groups * (ks + 1) / KS; // this wavefront's share

  // Filter rows: piece p of 16 bytes is piece p % PIECES of channel p / PIECES.  (A channel past the end reads the last one's
  // row and is not stored; groups past the share are loaded and not used.)
  float *mine = smem + ks * kRows;
  int woff[St::LOADS];
#pragma unroll
  for (int i = 0; i < St::LOADS; i++) {
    const int p = i * 64 + lane, oc = p / St::PIECES;
    woff[i] = oc < 32 ? ((oc0 + oc < OC ? oc : OC - 1 - oc0) * g.IC * KK + St::PIECE * (p - oc * St::PIECES)) * 4 : kOutside;
  }
  typedef float Piece __attribute__((ext_vector_type(St::PIECE)));
  Piece stage[St::LOADS];
  auto load = [&](int group) {
#pragma unroll
    for (int i = 0; i < St::LOADS; i++)
      if constexpr (St::PIECE == 4) stage[i] = __builtin_bit_cast(Piece, __builtin_amdgcn_raw_buffer_load_b128(filter, woff[i], group * (2 * HALF * KK * 4), 0));
      else stage[i] = __builtin_bit_cast(Piece, __builtin_amdgcn_raw_buffer_load_b64(filter, woff[i], group * (2 * HALF * KK * 4), 0));
  };
  auto keep = [&]() {
#pragma unroll
    for (int i = 0; i < St::LOADS; i++) {
      const int p = i * 64 + lane, oc = p / St::PIECES;
      if (64 * (i + 1) <= 32 * St::PIECES || oc < 32) *reinterpret_cast<Piece *>(mine + oc * St::PITCH + St::PIECE * (p - oc * St::PIECES)) = stage[i];
    }
  };
  // The reduction walks units - a group, or one of its window rows - in a pipeline two deep: a unit's taps fly under the
  // matrix instructions of the one before.
  auto fetch = [&](float (&b)[STEPS], int group, int unit) {
    const unsigned out = (rowOut << unit) & 0x80000000u;
    const int down = unit * g.DH * g.W * 4;
#pragma unroll
    for (int i = 0; i < STEPS; i++) {
      const int at = WIN == 7 ? (int)((unsigned)(voff[i] + down) | out) : voff[WIN == 1 ? 0 : unit * STEPS + i];
      b[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(image, at, (group * (2 * HALF) + (WIN == 1 ? i : 0)) * HW4, 0));
    }
  };
  const float *ap = mine + l32 * St::PITCH + hl * (HALF * KK);
  auto multiply = [&](const float (&b)[STEPS], int inChunk, int unit) {
#pragma unroll
    for (int i = 0; i < STEPS; i++)
      acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(ap[inChunk * (2 * HALF * KK) + unit * STEPS + i], b[i], acc[0], 0, 0, 0);
  };
  constexpr int NU = St::CG * UNITS, TURN = NU % 2 ? 2 : 1; // units of a chunk; chunks until a unit's buffer is the first again
  float b[2][STEPS];
  if (g0 < g1) {
    load(g0);
    fetch(b[0], g0, 0);
  }
  for (int turn = g0; turn < g1; turn += TURN * St::CG) {
#pragma unroll
    for (int h = 0; h < TURN; h++) {
      const int chunk = turn + h * St::CG;
      if (h && chunk >= g1) break; // (uniform)
      keep();
      if (chunk + St::CG < g1) load(chunk + St::CG);
#pragma unroll
      for (int u = 0; u < NU; u++) {
        const int group = chunk + u / UNITS;
        if (u % UNITS == 0 && group >= g1) break; // (uniform)
        const int next = u + 1; // (fetched if it is still in the share)
        if (chunk + next / UNITS < g1) fetch(b[(h * NU + next) % 2], chunk + next / UNITS, next % UNITS);
        multiply(b[(h * NU + u) % 2], u / UNITS, u % UNITS);
      }
    }
  }
  if (KS > 1) __syncthreads(); // the partial sums take the filter rows' place
  auto &partial = *reinterpret_cast<float(*)[KS][16 * 64]>(smem);
  finishTile<1, KS, uint32_t>(acc, partial, 0, ks, bias, add, y, OC, P, oc0, nFirst, img, pix, lane, relu);
}

// ---- few taps -----------------------------------------------------------------------------
// A reduction of at most 2 NS taps (a network's stem: 3 channels, 3 x 3).  A wavefront keeps the
// filter of its OCT x 32 channels in registers, lane half hl the taps 2 s + hl of step s, and walks
// over tiles of 32 pixels; the taps of the next tile are in flight while this one's are multiplied
// and stored.
enum class Output { Cached, Through, Streamed, Added }; // plain stores, written through to memory, non-temporal; plain with an addend
template <int OCT, int NS, Output OUT>
__global__ __launch_bounds__(256, 2) void conv_few_taps_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                               const float *__restrict__ bias, float *__restrict__ y, ConvGeo g, int OC,
                                                               int P, int N, FastDiv byP, FastDiv byOW, const float *__restrict__ add,
                                                               int relu, int K, int tiles, int tileStep) {
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int l32 = lane % 32, hl = lane / 32;
  const int oc0 = blockIdx.y * (32 * OCT);
  const int pixels = N * P;

  // Filter values, and where the lane half's tap of each step sits: its byte offset from the pixel's
  // first tap and its window position (kw | kh << 5; 31 past the end, a column that is always outside).
  float a[OCT][NS];
  int toff[NS], tpos[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) {
    const int k = 2 * s + hl;
    const int ic = k / (g.KW * g.KH), r = k - ic * (g.KW * g.KH);
    const int kh = r / g.KW, kw = r - kh * g.KW;
    const bool in = k < K;
    toff[s] = in ? ((ic * g.H + kh * g.DH) * g.W + kw * g.DW) * 4 : 0;
    tpos[s] = in ? kw | kh << 5 : 31;
#pragma unroll
    for (int t = 0; t < OCT; t++) {
      const int oc = oc0 + 32 * t + l32 < OC ? oc0 + 32 * t + l32 : OC - 1;
      const float v = w[(int64_t)oc * K + (in ? k : 0)];
      a[t][s] = in ? v : 0.0f;
    }
  }

  struct Tile {
    int pix, img, nFirst; // the lane's pixel (-1: past the end), its image less the tile's first, that image
    float b[NS];
  };
  const int64_t imageElems = (int64_t)g.IC * g.H * g.W;
  auto fetch = [&](Tile &o, int tile) {
    const int q0 = tile * 32, q = q0 + l32;
    const bool live = q < pixels;
    o.nFirst = __builtin_amdgcn_readfirstlane(divide(q0, byP));
    const int n = live ? divide(q, byP) : o.nFirst;
    const int p = live ? q - n * P : 0;
    const int oh = divide(p, byOW), ow = p - oh * g.OW;
    o.img = n - o.nFirst;
    o.pix = live ? p : -1;
    const int ih0 = oh * g.SH - g.PHL, iw0 = ow * g.SW - g.PWL;
    const unsigned rowOut = live ? outsideBits(ih0, g.H, g.KH, g.DH) : ~0u;
    const unsigned colOut = outsideBits(iw0, g.W, g.KW, g.DW) | 0x80000000u;
    const int base = (o.img * (int)imageElems + ih0 * g.W + iw0) * 4;
    const auto rsrc = resource(x + o.nFirst * imageElems, (N - o.nFirst) * imageElems);
#pragma unroll
    for (int s = 0; s < NS; s++) {
      const int out = __builtin_amdgcn_sbfe(rowOut, tpos[s] >> 5, 1) | __builtin_amdgcn_sbfe(colOut, tpos[s], 1);
      o.b[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (base + toff[s]) | out, 0, 0));
    }
  };
  float bv[OCT][16]; // the accumulators start from the bias
#pragma unroll
  for (int t = 0; t < OCT; t++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int oc = oc0 + 32 * t + 8 * (r / 4) + r % 4 + 4 * hl;
      bv[t][r] = bias[oc < OC ? oc : OC - 1];
    }
  const bool fullOc = oc0 + 32 * OCT <= OC;
  const int64_t outElems = (int64_t)OC * P;
  auto finish = [&](Tile &o) {
    // (stores through the bounds check too: a pixel or a channel past the end is dropped by it)
    const auto out = resource(y + o.nFirst * outElems, (N - o.nFirst) * outElems);
    const int at = o.pix < 0 ? kOutside : ((o.img * OC + oc0 + 4 * hl) * P + o.pix) * 4;
    // (opaque, or the compiler keeps their multiples and comparisons in scalar registers across the loop)
    int row = P * 4, channels = OC;
    asm volatile("" : "+s"(row), "+s"(channels));
    auto everyChannel = [&](auto each) { // of the lane: its register, its byte offsets
      if (fullOc) {
#pragma unroll
        for (int t = 0; t < OCT; t++)
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const int ocl = 32 * t + 8 * (r / 4) + r % 4;
            each(t, r, at, ocl * row);
          }
      } else {
#pragma unroll
        for (int t = 0; t < OCT; t++)
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const int ocl = 32 * t + 8 * (r / 4) + r % 4;
            if (oc0 + ocl < channels) // (a scalar offset past the resource would wrap the check)
              each(t, r, oc0 + ocl + 4 * hl < channels ? at : kOutside, ocl * row);
          }
      }
    };
    // (the addend is in flight under the matrix instructions: loaded channel by channel between the stores, each load
    // waited for the stores before it; 8 x 3 x 224 x 224 -> 64 of stride 2 32.1 -> 17.0 us, 6 x 1 x 12 x 91 -> 256 7.0 -> 5.3)
    float addend[OCT][16];
    if (OUT == Output::Added) {
      const auto post = resource(add + o.nFirst * outElems, (N - o.nFirst) * outElems);
      everyChannel([&](int t, int r, int voffset, int soffset) {
        addend[t][r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(post, voffset, soffset, 0));
      });
    }
    f32x16 acc[OCT];
#pragma unroll
    for (int t = 0; t < OCT; t++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[t][i] = bv[t][i];
#pragma unroll
    for (int s = 0; s < NS; s++)
#pragma unroll
      for (int t = 0; t < OCT; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t][s], o.b[s], acc[t], 0, 0, 0);
    everyChannel([&](int t, int r, int voffset, int soffset) {
      const float v = OUT == Output::Added ? acc[t][r] + addend[t][r] : acc[t][r];
      // cuDNN's ReLU with CUDNN_NOT_PROPAGATE_NAN maps NaN to 0, as fmaxf does
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, relu ? fmaxf(v, 0.0f) : v), out, voffset, soffset,
                                            OUT == Output::Through ? 16 : 0);
    });
  };
  Tile even, odd;
  int tile = (int)blockIdx.x * 4 + wave;
  if (tile < tiles) fetch(even, tile);
  for (; tile < tiles; tile += 2 * tileStep) {
    if (tile + tileStep < tiles) fetch(odd, tile + tileStep);
    finish(even);
    if (tile + tileStep >= tiles) break;
    if (tile + 2 * tileStep < tiles) fetch(even, tile + 2 * tileStep);
    finish(odd);
  }
}

// ---- few taps, four pixels a lane ------------------------------------------------------------
// The same reduction where output rows are whole quads of pixels and the window's columns are neighbours.  Column l of
// accumulator j is pixel 4 l + j of a tile of 128, so that a lane holds four consecutive pixels of every channel of its
// registers: a store writes 16 bytes a lane, 512 of each of two channels, where pixel l of every accumulator gave 4 and
// 128.  And the taps of four neighbours overlap: a lane half takes whole window rows - NR of the IC * KH, the lower half the
// first - and per row one 16-byte load of the quad's own columns and KW - 1 single ones beside it serve 4 KW taps.
// What bounds it: the output and, not wholly hidden behind it, the matrix cores (15 steps of 64 clocks a 32 x 32 tile).  16 x 3 x
// 256 x 256 -> 64, 268 MB: 76.9 -> 65.5 us (1 x 1 from the same: 68.0 -> 49.2; a fill of as many bytes takes 39); 8 x 3 x 224 x
// 224 -> 64 with a postAdd 87 -> 49; 8 x 3 x 128 x 128 -> 16 11.0 -> 6.7.  Stores of one tile dealt out between the matrix
// instructions of the next measured the same, an order of tiles by XCD too, runs of tiles a wavefront 90.
// SPLIT: the products by the bf16 matrix instructions, operands taken apart into three numbers as in conv_split.hip: twelve steps of
// 32 clocks instead of 15 of 64, and fewer roundings (K = 27: error against 64 bits 1.1e-7 -> 0.39e-7; of a product without others, where the
// fp32 instructions round once, 0.6e-7 -> 1.6e-7 at most).  A tile with values so large that
// they or their sums might be none in pieces is done again behind the others, and what is no number takes the fp32 instructions'
// result.  us, fp32 instructions / this, outputs in turn: 16 x 3 x 256 x 256 -> 64 56.2 / 55.0, 16 x 3 x 224 x 224 -> 64 56.1 / 48.4, 4 x 3 x 224 x 224 -> 64 16.0 /
// 12.9, 16 x 3 x 76 x 248 -> 33 18.8 / 13.3, 8 x 1 x 112 x 112 -> 64, 5 x 5, 10.6 / 8.4; of two channels 16.9 / 16.4 (16 x 2 x 128 x 128 -> 64).  Each of the four
// pixels' taps taken apart for itself: 56.7, 50.6, 13.5, 14.7, 8.6, 16.3.
template <int KW, int NR, Output OUT, bool ADDED, bool SPLIT>
__global__ __launch_bounds__(256, 2) void conv_quads_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                            const float *__restrict__ bias, float *__restrict__ y, ConvGeo g, int OC,
                                                            int P, int N, FastDiv byP, FastDiv byOW, const float *__restrict__ add,
                                                            int relu, int tiles, int tileStep) {
  constexpr int SIDE = KW - 1; // columns beside the quad's own
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int l32 = lane % 32, hl = lane / 32;
  const int oc0 = blockIdx.y * 32;
  const int pixels = N * P, rows = g.IC * g.KH;

  float a[NR][KW];
  int toff[NR], tkh[NR]; // a row's byte offset from the quad's first tap, and its window row (31: past the end, always outside)
#pragma unroll
  for (int i = 0; i < NR; i++) {
    const int r = hl * NR + i, ic = r / g.KH, kh = r - ic * g.KH;
    const bool in = r < rows;
    toff[i] = in ? (ic * g.H + kh * g.DH) * g.W * 4 : 0;
    tkh[i] = in ? kh : 31;
  }
  auto loadFilter = [&]() { // the lane's channel, rows of its half
    const int oc = oc0 + l32 < OC ? oc0 + l32 : OC - 1;
#pragma unroll
    for (int i = 0; i < NR; i++) {
      const int r = hl * NR + i;
#pragma unroll
      for (int k = 0; k < KW; k++) a[i][k] = r < rows ? w[((int64_t)oc * rows + r) * KW + k] : 0.0f;
    }
  };
  loadFilter();
  float bv[16];
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int oc = oc0 + 8 * (r / 4) + r % 4 + 4 * hl;
    bv[r] = bias[oc < OC ? oc : OC - 1];
  }
  // SPLIT: the lane half's taps as eight each of STEPS matrix instructions, in pieces: of every row the pairs of neighbours, then the last
  // ones of two rows at a time.
  constexpr int TAPS = NR * KW, STEPS = (TAPS + 7) / 8, PAIRS = KW / 2;
  u32x4 ap[kPieces][STEPS];
  float most = 0.0f; // pixels below this are finite in pieces, and so are their sums (uniform)
  auto inOrder = [&](u32x4 (&piece)[kPieces][STEPS], auto &&pair, auto &&lasts) { // pair(row, first column), lasts(row, the next one or -1)
#pragma unroll
    for (int i = 0; i < 4 * STEPS; i++) {
      constexpr int OF_ROWS = NR * PAIRS;
      const int r = 2 * (i - OF_ROWS);
      uint32_t p[kPieces] = {0u, 0u, 0u};
      if (i < OF_ROWS) pair(p, i / PAIRS, i % PAIRS * 2);
      else if (r < NR) lasts(p, r, r + 1 < NR ? r + 1 : -1);
#pragma unroll
      for (int k = 0; k < kPieces; k++) piece[k][i / 4][i % 4] = p[k];
    }
  };
  if constexpr (SPLIT) {
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < TAPS; i++) m = fmaxf(m, fabsf(a[i / KW][i % KW]));
    m = group_max<64>(m);
    if (m < 0x1p100f) most = fminf(0x1p100f, 0x1p74f / fmaxf(m, 0x1p-26f)); // (32 products of less than 2^74 and two scales of 2^24)
    inOrder(ap, [&](uint32_t (&p)[kPieces], int row, int k) { splitTriple(a[row][k] * kSplitScale, a[row][k + 1] * kSplitScale, p); },
            [&](uint32_t (&p)[kPieces], int row, int next) {
              splitTriple(a[row][KW - 1] * kSplitScale, next < 0 ? 0.0f : a[next < 0 ? 0 : next][KW - 1] * kSplitScale, p);
            });
  }
  struct Tile {
    int pix, img, nFirst; // the lane's first pixel (-1: past the end), its image less the tile's first, that image
    f32x4 own[NR];        // of a row: the quad's own columns, those left of them, those right
    float side[NR][SIDE > 0 ? SIDE : 1];
  };
  const int64_t imageElems = (int64_t)g.IC * g.H * g.W;
  auto fetch = [&](Tile &o, int tile) {
    const int q0 = tile * 128, q = q0 + 4 * l32;
    const bool live = q < pixels;
    o.nFirst = __builtin_amdgcn_readfirstlane(divide(q0, byP));
    const int n = live ? divide(q, byP) : o.nFirst;
    const int p = live ? q - n * P : 0;
    const int oh = divide(p, byOW), ow = p - oh * g.OW;
    o.img = n - o.nFirst;
    o.pix = live ? p : -1;
    const int ih0 = oh * g.SH - g.PHL;
    const unsigned rowOut = live ? outsideBits(ih0, g.H, g.KH, g.DH) | 0x80000000u : ~0u;
    const int base = (o.img * (int)imageElems + ih0 * g.W + ow) * 4; // of the quad's own columns
    const auto rsrc = resource(x + o.nFirst * imageElems, (N - o.nFirst) * imageElems);
    int sideOut[SIDE > 0 ? SIDE : 1], sideOff[SIDE > 0 ? SIDE : 1]; // column e of the window's KW + 3 is ow - PWL + e
#pragma unroll
    for (int e = 0; e < SIDE; e++) {
      const int d = e < g.PWL ? e - g.PWL : e - g.PWL + 4;
      sideOff[e] = d * 4;
      sideOut[e] = (unsigned)(ow + d) < (unsigned)g.W ? 0 : kOutside;
    }
#pragma unroll
    for (int i = 0; i < NR; i++) {
      const int out = __builtin_amdgcn_sbfe(rowOut, tkh[i], 1) & kOutside; // (not all ones: 16 bytes from there would wrap)
      o.own[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (base + toff[i]) | out, 0, 0));
#pragma unroll
      for (int e = 0; e < SIDE; e++)
        o.side[i][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (base + toff[i] + sideOff[e]) | out | sideOut[e], 0, 0));
    }
  };
  const int64_t outElems = (int64_t)OC * P;
  bool rest = false; // SPLIT: may there be sums that are no numbers in pieces? (uniform)
  auto finish = [&](Tile &o, auto againTag) {
    constexpr bool AGAIN = decltype(againTag)::value;
    const auto out = resource(y + o.nFirst * outElems, (N - o.nFirst) * outElems);
    const int at = o.pix < 0 ? kOutside : ((o.img * OC + oc0 + 4 * hl) * P + o.pix) * 4;
    int row = P * 4, channels = OC;
    asm volatile("" : "+s"(row), "+s"(channels));
    auto everyChannel = [&](auto each) { // of the lane: its register, its byte offsets
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int ocl = 8 * (r / 4) + r % 4;
        if (oc0 + ocl >= channels) break; // (uniform; a scalar offset past the resource would wrap the check)
        each(r, oc0 + ocl + 4 * hl < channels ? at : kOutside, ocl * row);
      }
    };
    // The addend: in flight under the matrix instructions (16 x 3 x 256 x 256 -> 64 140 -> 126 us, 8 x 1 x 128 x 128 -> 96, 5 x 5,
    // 27.1 -> 22.0), where the registers last: NR = 8 loads it a channel at a time (8 x 16 x 128 x 128 -> 64 15.8, so 21.6).
    constexpr bool kEarly = NR < 8;
    const auto post = resource(add + (ADDED ? o.nFirst * outElems : 0), (N - o.nFirst) * outElems);
    auto fromPost = [&](int voffset, int soffset) {
      return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(post, voffset, soffset, 0));
    };
    f32x4 addend[16];
    if (ADDED && kEarly) everyChannel([&](int r, int voffset, int soffset) { addend[r] = fromPost(voffset, soffset); });
    // the window's KW + 3 columns of a row in order (uniform selects: PWL of them lie left of the quad)
    auto columns = [&](int i, float (&c)[KW + 3]) {
#pragma unroll
      for (int e = 0; e < KW + 3; e++) {
        float v = e < SIDE ? o.side[i][e] : 0.0f; // e < PWL
#pragma unroll
        for (int own = 0; own < 4; own++)
          if (e - own >= 0 && e - own <= SIDE && e - own == g.PWL) v = o.own[i][own];
        if (e >= 4 && e - 4 >= 0 && e - 4 < SIDE && e >= g.PWL + 4) v = o.side[i][e - 4];
        c[e] = v;
      }
    };
    auto store = [&](const f32x16 (&acc)[4]) {
      everyChannel([&](int r, int voffset, int soffset) {
        f32x4 v = {acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
        if (ADDED) v += kEarly ? addend[r] : fromPost(voffset, soffset);
        // cuDNN's ReLU with CUDNN_NOT_PROPAGATE_NAN maps NaN to 0, as fmaxf does
        if (relu) v = f32x4{fmaxf(v[0], 0.0f), fmaxf(v[1], 0.0f), fmaxf(v[2], 0.0f), fmaxf(v[3], 0.0f)};
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), out, voffset, soffset,
                                               OUT == Output::Streamed ? 2 : OUT == Output::Through ? 16 : 0);
      });
    };
    f32x16 acc[4];
    if constexpr (SPLIT) {
      // Two columns at a time are taken apart, once for the four pixels; what starts at an odd one is put together from halves.
      float c[NR][KW + 3], m = 0.0f;
      uint32_t two[NR][(KW + 3) / 2][kPieces];
#pragma unroll
      for (int i = 0; i < NR; i++) {
        columns(i, c[i]);
#pragma unroll
        for (int e = 0; e < KW + 3; e++) m = fmaxf(m, fabsf(c[i][e]));
#pragma unroll
        for (int e = 0; e < KW + 3; e += 2) splitTriple(c[i][e] * kSplitScale, c[i][e + 1] * kSplitScale, two[i][e / 2]);
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        u32x4 bp[kPieces][STEPS];
        inOrder(bp,
                [&](uint32_t (&p)[kPieces], int row, int k) {
#pragma unroll
                  for (int n = 0; n < kPieces; n++) {
                    const int e = k + j;
                    p[n] = e % 2 ? __builtin_amdgcn_alignbit(two[row][e / 2 + 1][n], two[row][e / 2][n], 16) : two[row][e / 2][n];
                  }
                },
                [&](uint32_t (&p)[kPieces], int row, int next) {
#pragma unroll
                  for (int n = 0; n < kPieces; n++) {
                    const int e = KW - 1 + j;
                    p[n] = __builtin_amdgcn_perm(next < 0 ? 0u : two[next < 0 ? 0 : next][e / 2][n], two[row][e / 2][n], e % 2 ? 0x07060302u : 0x05040100u);
                  }
                });
        f32x16 sum;
#pragma unroll
        for (int i = 0; i < 16; i++) sum[i] = 0.0f;
        // (the small products first: their roundings are small, too)
#pragma unroll
        for (int order = kPieces - 1; order >= 0; order--)
#pragma unroll
          for (int k = 0; k <= order; k++)
#pragma unroll
            for (int i = 0; i < STEPS; i++)
              sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ap[k][i]), __builtin_bit_cast(bf16x8, bp[order - k][i]), sum, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 16; i++) acc[j][i] = fmaf(sum[i], kSplitUnscale, bv[i]);
        __builtin_amdgcn_sched_barrier(0); // (one pixel after the other: 5 x 5 would spill)
      }
      const bool numbers = __builtin_amdgcn_ballot_w64(!(m < most)) == 0; // (a NaN is one in either way)
      if constexpr (AGAIN) {
        if (numbers) return;
#pragma unroll
        for (int j = 0; j < 4; j++) {
          f32x16 plain;
#pragma unroll
          for (int i = 0; i < 16; i++) plain[i] = bv[i];
#pragma unroll
          for (int i = 0; i < TAPS; i++) plain = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i / KW][i % KW], c[i / KW][i % KW + j], plain, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 16; i++) acc[j][i] = fabsf(acc[j][i]) < __builtin_inff() ? acc[j][i] : plain[i];
        }
      } else {
        rest |= !numbers;
      }
      store(acc);
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[j][i] = bv[i];
#pragma unroll
      for (int i = 0; i < NR; i++) {
        float c[KW + 3];
        columns(i, c);
#pragma unroll
        for (int k = 0; k < KW; k++)
#pragma unroll
          for (int j = 0; j < 4; j++) acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][k], c[k + j], acc[j], 0, 0, 0);
      }
      store(acc);
    }
  };
  Tile even, odd;
  int tile = (int)blockIdx.x * 4 + wave;
  if (tile < tiles) fetch(even, tile);
  for (; tile < tiles; tile += 2 * tileStep) {
    if (tile + tileStep < tiles) fetch(odd, tile + tileStep);
    finish(even, std::false_type());
    if (tile + tileStep >= tiles) break;
    if (tile + 2 * tileStep < tiles) fetch(even, tile + 2 * tileStep);
    finish(odd, std::false_type());
  }
  if constexpr (SPLIT) {
    if (!rest) return;
    loadFilter(); // (here, where the operands of the fp32 instructions cost the loop above no registers)
    for (tile = (int)blockIdx.x * 4 + wave; tile < tiles; tile += tileStep) {
      fetch(even, tile);
      finish(even, std::true_type());
    }
  }
}

// ---- larger windows over few channels -----------------------------------------------------------
// A stem: 5 x 5 or 7 x 7 from one channel or three, 49 to 147 taps.  The window kernel reads a tap a lane from memory for every
// matrix instruction and pairs channels, of which one or three leave a quarter or half for nothing (8 x 3 x 224 x 224 -> 64, 7 x 7
// of stride 2: 44 us, 13 by the matrix cores; now 30).  Here a tile is 32 neighbouring pixels of one output row, and the input under it
// - IC * KH window rows of 31 SW + KW columns - comes in whole lines into an LDS patch of the wavefront's own, each element
// once, with zeros where the window leaves the image, while the tile before is multiplied.  Lane half hl takes window rows
// hl * NR and on, so that a step's taps lie at one immediate offset from the lane's place in the patch; the filter lies in LDS in the
// order of the steps.  The loop is LDS reads and matrix instructions, nothing else.
template <int KW, int NR, int SW, bool ADDED>
__global__ __launch_bounds__(256, 2) void conv_patch_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                            const float *__restrict__ bias, float *__restrict__ y, ConvGeo g, int OC, int P,
                                                            int N, FastDiv byAcross, FastDiv byOH, const float *__restrict__ add, int relu,
                                                            int across, int tiles, int tileStep) {
  constexpr int COLS = 31 * SW + KW, LOADS = (2 * NR * COLS + 63) / 64, STEPS = NR * KW;
  constexpr int PITCH = 33;                // channels of a step, apart for the writes along the steps
  __shared__ float filter[STEPS * 2 * PITCH]; // [step][lane half][channel]
  __shared__ float patches[4][LOADS * 64];
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int l32 = lane % 32, hl = lane / 32;
  const int oc0 = blockIdx.y * 32, rows = g.IC * g.KH;
  constexpr int FILL = (STEPS * 2 * 32 + 255) / 256;
  float fill[FILL]; // (all in flight at once)
  const auto weights = resource(w + (int64_t)oc0 * (rows * KW), (int64_t)(OC - oc0) * (rows * KW));
#pragma unroll
  for (int i = 0; i < FILL; i++) {
    const int e = i * 256 + tid, oc = e / (2 * STEPS), k = e - oc * (2 * STEPS);
    fill[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(weights, k < rows * KW ? (oc * (rows * KW) + k) * 4 : kOutside, 0, 0));
  }
#pragma unroll
  for (int i = 0; i < FILL; i++) {
    const int e = i * 256 + tid, oc = e / (2 * STEPS), k = e - oc * (2 * STEPS), half = k / STEPS;
    if (oc < 32) filter[((k - half * STEPS) * 2 + half) * PITCH + oc] = fill[i];
  }
  float bv[16]; // the accumulators start from the bias
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int oc = oc0 + 8 * (r / 4) + r % 4 + 4 * hl;
    bv[r] = bias[oc < OC ? oc : OC - 1];
  }
  // Element i * 64 + lane of the patch: its byte offset from the tile's first tap (kOutside past the last window row), column and row
  // in the window.
  int poff[LOADS], pcol[LOADS], prow[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; i++) {
    const int e = i * 64 + lane, r = e / COLS, c = e - r * COLS, ic = r / KW, kh = r - ic * KW;
    poff[i] = r < rows ? ((ic * g.H + kh * g.DH) * g.W + c) * 4 : kOutside;
    pcol[i] = r < rows ? c : 1 << 30; // (always outside: an offset from kOutside could wrap)
    prow[i] = kh;
  }
  float *patch = patches[wave];
  const int64_t imageElems = (int64_t)g.IC * g.H * g.W, outElems = (int64_t)OC * P;
  float next[LOADS];
  struct Place {
    int n, oh, ow0;
  };
  auto place = [&](int tile) {
    const int row = divide(tile, byAcross), n = divide(row, byOH);
    return Place{n, row - n * g.OH, (tile - row * across) * 32};
  };
  auto fetch = [&](int tile) {
    const Place o = place(tile);
    const int ih0 = o.oh * g.SH - g.PHL, iw0 = o.ow0 * SW - g.PWL;
    const unsigned rowOut = outsideBits(ih0, g.H, KW, g.DH) & ((1u << KW) - 1u);
    const auto rsrc = resource(x + o.n * imageElems, (N - o.n) * imageElems);
    const int first = (ih0 * g.W + iw0) * 4;
    if (iw0 >= 0 && iw0 + COLS <= g.W && !rowOut) { // (uniform) nothing outside
#pragma unroll
      for (int i = 0; i < LOADS; i++) next[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, poff[i], first, 0));
    } else {
#pragma unroll
      for (int i = 0; i < LOADS; i++) {
        const bool in = (unsigned)(iw0 + pcol[i]) < (unsigned)g.W;
        const int out = __builtin_amdgcn_sbfe(rowOut, prow[i], 1) & kOutside;
        next[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, in ? (first + poff[i]) | out : kOutside, 0, 0));
      }
    }
  };
  auto keep = [&]() {
#pragma unroll
    for (int i = 0; i < LOADS; i++) patch[i * 64 + lane] = next[i];
  };
  const bool fullOc = oc0 + 32 <= OC;
  const float *ap = filter + hl * PITCH + l32, *bp = patch + hl * (NR * COLS) + l32 * SW;
  int tile = (int)blockIdx.x * 4 + wave;
  if (tile < tiles) {
    fetch(tile);
    keep();
  }
  __syncthreads(); // the filter
  for (; tile < tiles; tile += tileStep) {
    const bool more = tile + tileStep < tiles;
    if (more) fetch(tile + tileStep);
    const Place o = place(tile);
    const auto out = resource(y + o.n * outElems, (N - o.n) * outElems);
    const int at = o.ow0 + l32 < g.OW ? ((oc0 + 4 * hl) * P + o.oh * g.OW + o.ow0 + l32) * 4 : kOutside;
    int row = P * 4, channels = OC;
    asm volatile("" : "+s"(row), "+s"(channels));
    auto everyChannel = [&](auto each) { // of the lane: its register, its byte offsets
      if (fullOc) {
#pragma unroll
        for (int r = 0; r < 16; r++) each(r, at, (8 * (r / 4) + r % 4) * row);
      } else {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int ocl = 8 * (r / 4) + r % 4;
          if (oc0 + ocl < channels) // (a scalar offset past the resource would wrap the check)
            each(r, oc0 + ocl + 4 * hl < channels ? at : kOutside, ocl * row);
        }
      }
    };
    float addend[16]; // (in flight under the matrix instructions)
    if (ADDED) {
      const auto post = resource(add + o.n * outElems, (N - o.n) * outElems);
      everyChannel([&](int r, int voffset, int soffset) {
        addend[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(post, voffset, soffset, 0));
      });
    }
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; i++) acc[i] = bv[i];
    // One window row's operands are read under the matrix instructions of the row before (the fences keep them there).
    float av[2][KW], bw[2][KW];
    auto read = [&](int i) {
#pragma unroll
      for (int k = 0; k < KW; k++) {
        bw[i % 2][k] = bp[i * COLS + k];
        av[i % 2][k] = ap[(i * KW + k) * (2 * PITCH)];
      }
    };
    read(0);
#pragma unroll
    for (int i = 0; i < NR; i++) {
      if (i + 1 < NR) read(i + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < KW; k++)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i % 2][k], bw[i % 2][k], acc, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    everyChannel([&](int r, int voffset, int soffset) {
      const float v = ADDED ? acc[r] + addend[r] : acc[r];
      // cuDNN's ReLU with CUDNN_NOT_PROPAGATE_NAN maps NaN to 0, as fmaxf does
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, relu ? fmaxf(v, 0.0f) : v), out, voffset, soffset, 16);
    });
    if (more) keep();
  }
}

// ---- square windows, operands shared through LDS ---------------------------------------------
// A block owns 64 output channels x 64 output pixels: 2 x 2 wavefronts of a 32 x 32 tile each, KS
// times over when KS groups of four wavefronts split the channel groups.  Per unit of a channel group
// its taps and filter values go from memory straight into LDS (dword loads; the bounds check writes
// the zeros) into a ring of three stages, two units ahead of the one multiplied, the loads dealt out
// between the MFMAs.  Every byte from L2 feeds 64 channels or pixels instead of the window kernel's
// 32, whose L2 traffic is what bounds that one on large grids (8 x 256 x 14 x 14 -> 512, 3 x 3: 70 us
// there, 45 here).
template <int WIN, int KS>
__global__ __launch_bounds__(256 * KS, 2) void conv_tile_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                                const float *__restrict__ bias, float *__restrict__ y, ConvGeo g,
                                                                int OC, int P, int N, FastDiv byP, FastDiv byOW,
                                                                const float *__restrict__ add, int relu) {
  using Win = Window<WIN>;
  constexpr int KK = Win::KK, UNITS = Win::UNITS, STEPS = Win::STEPS, HALF = Win::HALF;
  constexpr int TL = (STEPS + 1) / 2;         // tap loads per wavefront and unit: every other step of one channel half
  constexpr int PITCH = 18;                   // words per channel of the filter slice (2 * STEPS of them used; even, so that 32 channels fall on 32 banks)
  constexpr int WL = 5;                       // filter loads per wavefront and unit: 4 x 5 x 64 >= 64 x PITCH
  constexpr int ND = TL + WL;                 // loads per wavefront and unit
  constexpr int kTapWords = 2 * TL * 2 * 64;  // [step][half][pixel]
  constexpr int kStageWords = kTapWords + 4 * WL * 64;
  constexpr int kRing = 3;
  constexpr int kLds = KS * kRing * kStageWords * 4;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[kLds];
  static_assert(KS == 1 || KS * 4 * 4096 <= kLds, "the partial sums take the ring's place");

  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int l32 = lane % 32, hl = lane / 32;
  const int ks = wave / 4, wv = wave % 4;
  const int wm = wv / 2, wp = wv % 2; // 32-channel and 32-pixel half of the block's tile
  const int oc0 = blockIdx.y * 64, q0 = pixelBlock<256 * KS>() * 64;
  const int HW4 = g.H * g.W * 4, pixels = N * P;
  if (q0 >= pixels) return;
  const int nFirst = __builtin_amdgcn_readfirstlane(divide(q0, byP));

  // ---- movers.  Wavefront wv moves channel half wv / 2 of the taps, the steps of parity wv % 2.  The
  // upper half's pixels are kept with bit 5 flipped, so that the two halves a wavefront reads at once lie
  // on different banks.
  const int mhalf = wv / 2, mstep = wv % 2;
  int voff[UNITS * TL];
  {
    const int q = q0 + (lane ^ (32 * mhalf));
    const bool live = q < pixels;
    const int n = live ? divide(q, byP) : nFirst;
    const int p = live ? q - n * P : 0;
    const int oh = divide(p, byOW), ow = p - oh * g.OW;
    const int ih0 = live ? oh * g.SH - g.PHL : -kNever, iw0 = ow * g.SW - g.PWL;
    const int base = ((n - nFirst) * g.IC + mhalf * HALF) * HW4 + ((oh * g.SH - g.PHL) * g.W + iw0) * 4;
#pragma unroll
    for (int u = 0; u < UNITS; u++)
#pragma unroll
      for (int i = 0; i < TL; i++) {
        // (1 x 1: every step reads the same position of another channel)
        const int pos = WIN == 1 ? 0 : u * STEPS + 2 * i + mstep;
        const int kh = pos / WIN, kw = pos - kh * WIN;
        const bool in = (unsigned)(ih0 + kh * g.DH) < (unsigned)g.H && (unsigned)(iw0 + kw * g.DW) < (unsigned)g.W;
        voff[u * TL + i] = in ? base + (kh * g.DH * g.W + kw * g.DW) * 4 : kOutside;
      }
  }
  // The filter slice: word e = channel * PITCH + half * STEPS + step.
  int woff[WL], wch[WL]; // byte offset at group 0, unit 0; channel inside the group (beyond every group: nothing to fetch)
  {
    const int row = g.IC * (KK * 4); // bytes per output channel
    int oc = (WL * 64 * wv + lane) / PITCH, k = (WL * 64 * wv + lane) - oc * PITCH;
    int at = oc * row;
#pragma unroll
    for (int i = 0; i < WL; i++) { // the next load's word is 64 = 3 * PITCH + 10 further
      const bool upper = k >= STEPS;
      const bool used = oc < 64 && oc0 + oc < OC && k < 2 * STEPS;
      woff[i] = used ? at + k * 4 + (WIN > 1 && upper ? (KK - STEPS) * 4 : 0) : kOutside;
      wch[i] = !used ? 0x3fffffff : WIN == 1 ? k : upper ? 1 : 0;
      const bool wrap = k >= PITCH - 10;
      k += wrap ? 10 - PITCH : 10;
      oc += wrap ? 4 : 3;
      at += wrap ? 4 * row : 3 * row;
    }
  }
  const int64_t imageElems = (int64_t)g.IC * g.H * g.W;
  const i32x4 image = resourceWords(x + nFirst * imageElems, (N - nFirst) * imageElems);
  const i32x4 filter = resourceWords(w + (int64_t)oc0 * g.IC * KK, (int64_t)(OC - oc0) * g.IC * KK);
  const uint32_t ldsBase = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) unsigned char *)smem) + ks * (kRing * kStageWords * 4);
  // (inline assembly: completion is tracked by hand, see gemm_mfma.hip)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  auto dma4 = [&](int voffset, const i32x4 &rsrc, int soffset, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dword %0, %1, %2 offen lds"
                 :
                 : "v"(voffset), "s"(rsrc), "s"(soffset), "s"(lds)
                 : "memory", "m0");
  };
#pragma clang diagnostic pop

  const int groups = (g.IC + 2 * HALF - 1) / (2 * HALF);
  const int perKs = (groups + KS - 1) / KS; // every wavefront group walks as many; those past the end fetch zeros
  const int gBegin = ks * perKs;
  // Load k of the wavefront's for a unit.  `whole`: every channel of the group exists (uniform).
  auto load = [&](int k, int group, int unit, uint32_t at, auto whole) {
    const int c0 = group * (2 * HALF);
    if (k < TL) {
      const int step = 2 * k + mstep;
      const int c = c0 + (WIN == 1 ? step : 0); // the channel these 64 lanes read, less mhalf * HALF
      const bool in = step < STEPS && (decltype(whole)::value || c + mhalf * HALF < g.IC);
      dma4(in ? voff[unit * TL + k] : kOutside, image, in ? c * HW4 : 0, at + (uint32_t)((step * 2 + mhalf) * 64 * 4));
    } else {
      const int i = k - TL;
      const bool in = decltype(whole)::value || c0 + wch[i] < g.IC;
      // (a scalar offset beyond the resource would wrap the bounds check: 0 where nothing is in range)
      const int wbase = decltype(whole)::value || c0 < g.IC ? (c0 * KK + unit * STEPS) * 4 : 0;
      dma4(in ? woff[i] : kOutside, filter, wbase, at + (uint32_t)((kTapWords + (WL * wv + i) * 64) * 4));
    }
  };

  f32x16 acc[1];
#pragma unroll
  for (int i = 0; i < 16; i++) acc[0][i] = 0.0f;

  const int total = perKs * UNITS;
  auto unitOf = [&](int t, auto &&f) { // f(group, unit as a constant) of the t-th unit
    if constexpr (UNITS == 1) f(gBegin + t, std::integral_constant<int, 0>());
    else {
      const int grp = gBegin + t / UNITS, u = t % UNITS;
      auto pick = [&](auto self, auto c) {
        constexpr int k = decltype(c)::value;
        if constexpr (k < UNITS) {
          if (u == k) f(grp, c);
          else self(self, std::integral_constant<int, k + 1>());
        }
      };
      pick(pick, std::integral_constant<int, 0>());
    }
  };
  auto loadUnit = [&](int t, int stage, auto &&take) { // take(load index -> void) issues the loads of unit t
    unitOf(t, [&](int grp, auto u) {
      const uint32_t into = ldsBase + (uint32_t)stage * (kStageWords * 4);
      if ((grp + 1) * (2 * HALF) <= g.IC) take([&](int k) { load(k, grp, decltype(u)::value, into, std::true_type()); });
      else take([&](int k) { load(k, grp, decltype(u)::value, into, std::false_type()); });
    });
  };
  auto allAtOnce = [&](auto &&one) {
#pragma unroll
    for (int k = 0; k < ND; k++) one(k);
  };
  loadUnit(0, 0, allAtOnce);
  if (total > 1) loadUnit(1, 1, allAtOnce);
  // One unit: the MFMAs of its steps, each step's operands read from LDS one step ahead, and the
  // loads of a later unit dealt out between the steps.
  auto compute = [&](int stage, auto &&between) {
    const auto *at = reinterpret_cast<const float __attribute__((address_space(3))) *>((uintptr_t)(ldsBase + (uint32_t)stage * (kStageWords * 4)));
    const auto *ap = at + kTapWords + (32 * wm + l32) * PITCH + hl * STEPS;
    const auto *bp = at + hl * 64 + ((wp * 32 + l32) ^ (32 * hl));
    float a[2], b[2];
    a[0] = ap[0];
    b[0] = bp[0];
#pragma unroll
    for (int i = 0; i < STEPS; i++) {
      if (i + 1 < STEPS) {
        a[(i + 1) % 2] = ap[i + 1];
        b[(i + 1) % 2] = bp[(i + 1) * 2 * 64];
      }
      acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i % 2], b[i % 2], acc[0], 0, 0, 0);
      between(i);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int stage = 0;
  for (int t = 0; t < total; t++) {
    // unit t has landed (the one after may fly); everybody is done with unit t - 1, whose stage the
    // loads of unit t + 2 overwrite
    if (t + 1 < total) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(ND) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t + 2 < total)
      loadUnit(t + 2, stage >= 1 ? stage - 1 : stage + 2, [&](auto &&one) {
        compute(stage, [&](int i) {
#pragma unroll
          for (int k = i * ND / STEPS; k < (i + 1) * ND / STEPS; k++) one(k);
        });
      });
    else compute(stage, [](int) {});
    stage = stage == kRing - 1 ? 0 : stage + 1;
  }

  const int q = q0 + wp * 32 + l32;
  const bool live = q < pixels;
  const int n = live ? divide(q, byP) : nFirst;
  const int img[1] = {n - nFirst}, pix[1] = {live ? q - n * P : -1};
  if (KS > 1) __syncthreads(); // the partial sums take the ring's place
  auto &partial = *reinterpret_cast<float(*)[KS > 1 ? 4 * KS : 1][KS > 1 ? 16 * 64 : 1]>(smem);
  finishTile<1, KS, uint32_t>(acc, partial, wv * KS, ks, bias, add, y, OC, P, oc0 + 32 * wm, nFirst, img, pix, lane, relu);
}

// One output a thread.  Index: 32 bits where input and output allow (64-bit divisions are sequences of
// a hundred instructions, longer than the window's loads; 4 x 64 x 28 x 28, 2 x 2: 2.5 -> 2.1 us).
template <typename Index>
__global__ __launch_bounds__(256) void pool_kernel(const float *__restrict__ x, float *__restrict__ y, Index total, Index stride,
                                                   int H, int W, int OH, int OW, int KH, int KW, int PHL, int PWL, int SH,
                                                   int SW, bool average) {
  for (Index i = (Index)blockIdx.x * 256 + threadIdx.x; i < total; i += stride) {
    const Index row = i / OW; // output row over all planes
    const int ow = (int)(i - row * OW), oh = (int)(row % OH);
    const float *plane = x + (row / OH) * (Index)H * W;
    // the part of the window inside the image
    const int h0 = oh * SH - PHL, w0 = ow * SW - PWL;
    const int hFrom = h0 < 0 ? 0 : h0, hTo = h0 + KH < H ? h0 + KH : H;
    const int wFrom = w0 < 0 ? 0 : w0, wTo = w0 + KW < W ? w0 + KW : W;
    float acc = average ? 0.0f : -INFINITY;
    for (int ih = hFrom; ih < hTo; ih++)
      for (int iw = wFrom; iw < wTo; iw++) {
        const float v = plane[(Index)ih * W + iw];
        acc = average ? acc + v : fmaxf(acc, v);
      }
    y[i] = average ? acc / (float)(KH * KW) : acc;
  }
}

unsigned blocksFor(int64_t items) {
  int64_t blocks = (items + 255) / 256;
  if (blocks > kMaxStreamBlocks) blocks = kMaxStreamBlocks;
  return (unsigned)(blocks > 0 ? blocks : 1);
}

bool fitsInt(int64_t v) { return v >= 0 && v <= 0x7fffffff; }

} // namespace

// How many wavefronts share a tile of conv_staged_kernel, 0 where another kernel is faster.  By size eight or four are in question (us, what
// ran before / four / eight, 3 x 3 unless said otherwise): from 32 channel groups up to two tiles a CU (196 tiles of 32 groups 6.81 / - / 5.98,
// 112 of 128 20.8 / - / 16.8, 496 of 128 45.1 / 27.9 / 27.0), from 16 beyond 1.5 a CU, up to eight (1176 tiles of 96 channels 1.3 to
// 1.6 times as fast, 3136 tiles 28.0 / 29.7), up to three where the 64 x 64 tiles are the alternative (784 15.5 / 14.9, 980 48.2 / 48.5); 5 x 5, of whose blocks of
// eight a CU holds one, the same with half the groups (248 tiles of 32 16.5 / 13.5 / 12.0, 442 42.9 / 23.3 / 24.2); 7 x 7 from 8 groups (112 of 128
// 156 / 85 / 75).  1 x 1 gained nothing: sixteen channels of a row are one line already.
// Whether they gain is what an estimate says, of the logarithm of their time over the former kernel's, fitted to 2600 of 4000 shapes timed
// on all three: the more, the longer the reduction; the more channels a tile has, whose rows are the lines that an instruction of the other
// kernels touches; where a row of the filter is whole lines, since staged loads run along it; where taps lie apart, at a stride or
// in short rows; and the more of their last round the other kernels waste, which take two tiles a wavefront or 64 x 64.  (us, before / staged:
// 230 tiles from 64 channels 6.9 / 6.4, from 72 6.8 / 8.1; 16 channels from 128 9.1 / 9.7; 23 x 242 x 15 from 16 to 160, 5 x 5 of stride 2, 58 / 41.)
// Over the 4000 it is 0.857 of the time without them, 10 more than 6 % slower; staged everywhere in question it was 0.861, 174.
int convStagedWaves(int win, int64_t stride, int64_t pixels, int64_t IC, int64_t OC, int64_t OW, int64_t cus) {
  if (IC % 2 || win < 3) return 0;
  const int64_t ocTiles = (OC + 31) / 32, tiles = (pixels + 31) / 32 * ocTiles, groups = IC / 2, r = (tiles + cus - 1) / cus;
  const bool paired = (OC - 1) % 64 >= 32; // the 64 x 64 tiles go beyond 400
  int waves = 0;
  if (win == 7) waves = groups < 8 || (paired && r > 3) ? 0 : r == 1 ? 8 : 4;
  else if (tiles <= (win == 3 ? 2 * cus : cus) && groups >= (win == 3 ? 32 : 16)) waves = 8;
  else if (win == 3) waves = groups >= 16 && 2 * tiles > 3 * cus && r <= (paired ? 3 : 8) ? 4 : 0;
  else if (tiles > cus && (r <= 3 || !paired)) waves = groups >= (r == 4 ? 16 : 8) ? 4 : 0;
  if (!waves) return 0;
  // rounds of the CUs that the other kernels take, a tile each
  auto rounds = [&](int64_t blocks, int64_t each) { return (blocks + each * cus - 1) / (each * cus) * each; };
  const int64_t others = tiles <= 400 ? r : paired ? 4 * rounds((pixels + 63) / 64 * ((OC + 63) / 64), 1)
                                          : rounds(tiles, tiles <= 2048 ? 2 : win == 3 ? 8 : 4);
  static const double base[3][2] = {{0.341, 0.359}, {0.212, 0.238}, {0.190, 0.150}}; // 3 x 3, 5 x 5, 7 x 7; four, eight
  const double channels = (double)OC / (double)(32 * ocTiles), rows = std::min(4.0, 32.0 / (double)OW);
  const double change = base[(win - 3) / 2][waves / 8] - 0.071 * std::log((double)groups / 32.0) - 0.133 * std::log(channels) - (stride > 1 ? 0.039 : 0.0) -
                        0.011 * rows - (IC % 32 == 0 ? 0.099 : 0.0) - 0.318 * (double)others / (double)r;
  return change < -0.01 ? waves : 0;
}

// us that a 3 x 3 takes in the kernel that the lines of conv2d give it, where conv_split_kernel does not: each start + rounds of its tiles *
// (a part of its own + one a channel), fitted to 500 shapes (10th and 90th percentile 0.93 and 1.06 times what was measured; two
// groups of wavefronts on LDS tiles 0.79 and 0.98).
double convWindowTime(int64_t stride, int64_t pixels, int64_t IC, int64_t OC, int64_t OW, int64_t cus) {
  const int64_t tiles = (pixels + 31) / 32 * ((OC + 31) / 32), blocks = (pixels + 63) / 64 * ((OC + 63) / 64), units = (IC + 1) / 2;
  auto rounds = [](int64_t count, int64_t each) { return (double)((count + each - 1) / each); };
  const double channels = (double)IC;
  const int ks = convStagedWaves(3, stride, pixels, IC, OC, OW, cus);
  if (ks == 8) return 2.9 + rounds(tiles, cus) * (0.74 + 0.044 * channels);
  if (ks == 4) return 2.2 + rounds(tiles, cus) * (0.83 + 0.043 * channels);
  if (tiles <= 400) return 2.8 + rounds(tiles, cus) * 0.041 * channels;
  if ((OC - 1) % 64 >= 32) {
    if (blocks <= cus && units >= 64) return 7.0 + 0.156 * channels;
    if (blocks <= 2 * cus && units >= 24) return 3.0 + rounds(blocks, cus) * 0.155 * channels;
    return 4.75 + rounds(blocks, cus) * (0.65 + 0.159 * channels);
  }
  if (tiles <= 2048) return 3.0 + rounds(tiles, 2 * cus) * (0.67 + 0.087 * channels);
  return 2.6 + rounds(tiles, 8 * cus) * (1.33 + 0.319 * channels);
}

// us on few tiles, a closer fit there: 1100 launches of up to 325 tiles (10th and 90th percentile 0.81 to 0.93 and 1.06 to 1.10).
double convFewTilesTime(int win, int64_t stride, int64_t pixels, int64_t IC, int64_t OC, int64_t OW, int64_t cus) {
  const int64_t tiles = (pixels + 31) / 32 * ((OC + 31) / 32);
  const int ks = convStagedWaves(win, stride, pixels, IC, OC, OW, cus);
  if (ks == 4 || tiles > 400) return 0.0;
  const double rounds = (double)((tiles + cus - 1) / cus), channels = (double)IC;
  if (ks == 8) return win == 3 ? 3.6 + rounds * 0.0444 * channels : win == 5 ? 3.14 + rounds * (0.335 + 0.1305 * channels) : 2.65 + rounds * (0.97 + 0.275 * channels);
  return win == 3 ? 3.75 + rounds * 0.0355 * channels : win == 5 ? 3.56 + rounds * 0.131 * channels : 4.16 + rounds * 0.284 * channels;
}

// Do patches take a 5 x 5 or 7 x 7 from one channel or three?  From half of a row's tiles filled on (us, window tiles / patches, 7 x 7 from
// 3 channels unless said otherwise: 1 x 224 x 224 -> 64 of stride 2 13.0 / 7.4, 16 x 256 x 256 94 / 57, 4 x 112 x 112 -> 32 14.2 / 10.3, 2 x
// 28 x 28 -> 96 7.5 / 6.9; 32 x 28 x 28 -> 64 from 1 12.3 / 5.7; 5 x 5 16 x 128 x 128 -> 64 55 / 33; but rows of 10 13.1 / 16.4).  From one
// channel always.  From three, not where
//  * a 5 x 5 has few window tiles, whose start is shorter: up to one a CU (13 x 37 x 17 -> 24 5.5 / 6.0), at stride 2 up to 400, where they
//    take four wavefronts each (4 x 26 x 57 -> 32 5.0 / 5.9, 2 x 50 x 116 -> 24 5.3 / 6.1);
//  * half-filled rows cost patches another round of the SIMDs, a tile each, and the 64 x 64 tiles are no alternative: 8 x 95 x 146 -> 32, 5 x 5 of
//    stride 2, 6.4 / 7.6, 4 x 90 x 82 -> 8 8.4 / 9.5.
// Over 1500 shapes 0.82 of the time before, one more than 3 % slower, 1.06 times; without the last two lines 105 of 1300, up to 1.20 times.
bool convByPatches(int win, int stride, int64_t tiles, int64_t rowTiles, int64_t IC, int64_t OC, int64_t OW, int64_t cus) {
  if ((win != 5 && win != 7) || (IC != 1 && IC != 3) || stride > 2 || 2 * OW < (OW + 31) / 32 * 32) return false;
  if (IC == 1) return true;
  if (win == 5 && tiles <= (stride == 1 ? cus : 400)) return false;
  const int64_t simds = 4 * cus, rounds = (rowTiles + simds - 1) / simds, before = (tiles + simds - 1) / simds;
  const bool paired = (OC - 1) % 64 >= 32;
  return paired || 2 * rounds < (win == 5 && stride == 2 ? 3 : 4) * before;
}

void conv2d(const float *input, const float *weight, const float *bias, float *output, const float *postAdd,
            int64_t N, int64_t IC, int64_t H, int64_t W, int64_t OC, int64_t KH, int64_t KW, int64_t OH,
            int64_t OW, int64_t PHL, int64_t PWL, int64_t PHR, int64_t PWR, int64_t SH, int64_t SW, int64_t DH,
            int64_t DW, bool hasPostAdd, bool relu, hipStream_t stream) {
  if (N < 0 || IC <= 0 || H <= 0 || W <= 0 || OC <= 0 || KH <= 0 || KW <= 0 || OH < 0 || OW < 0)
    fail("mgpuConv2d: bad shape");
  if (PHL < 0 || PWL < 0 || PHR < 0 || PWR < 0 || SH <= 0 || SW <= 0 || DH <= 0 || DW <= 0)
    fail("mgpuConv2d: bad padding, stride or dilation");
  const int64_t spanH = H + PHL + PHR - DH * (KH - 1) - 1, spanW = W + PWL + PWR - DW * (KW - 1) - 1;
  if (spanH < 0 || spanW < 0 || OH != spanH / SH + 1 || OW != spanW / SW + 1)
    fail("mgpuConv2d: output size does not follow from input, kernel, padding, stride and dilation");
  if (N == 0) return;
  if (!input || !weight || !bias || !output) fail("mgpuConv2d: null pointer");
  if (hasPostAdd && !postAdd) fail("mgpuConv2d: hasPostAdd set but postAdd is null");
  const int64_t K = IC * KH * KW, P = OH * OW;
  for (int64_t v : {N, IC, H, W, OC, KH, KW, OH, OW, PHL, PWL, SH, SW, DH, DW, K, P, IC * H * W + (KH * DH + 1) * W + KW * DW})
    if (!fitsInt(v)) fail("mgpuConv2d: dimension too large");

  if (OH == 0 || OW == 0) return;
  const ConvGeo g{(int)IC, (int)H, (int)W, (int)KH, (int)KW, (int)OH, (int)OW, (int)PHL, (int)PWL,
                  (int)SH, (int)SW, (int)DH, (int)DW};
  const float *add = hasPostAdd ? postAdd : nullptr;
  const int64_t pixels = N * P, pix32 = (pixels + 31) / 32;
  const FastDiv byP = fastDiv((int)P), byOW = fastDiv((int)OW), byOH = fastDiv((int)OH);
  auto gridOf = [&](int64_t blocks, int64_t channels, int64_t threads) {
    const int64_t ocTiles = (OC + channels - 1) / channels;
    if (ocTiles > 65535) fail("mgpuConv2d: too many output channels for one launch");
    if (!fitsInt(blocks)) fail("mgpuConv2d: too many output tiles for one launch");
    if (blocks * threads < 2 * kGridRow) return dim3((unsigned)blocks, (unsigned)ocTiles);
    const int64_t row = kGridRow / threads;
    return dim3((unsigned)row, (unsigned)ocTiles, (unsigned)((blocks + row - 1) / row));
  };
  // Everything but the table kernel's wide form keeps pixel indices and, from the first image a tile
  // touches, byte offsets in 32 bits (a tile is at most 64 pixels), and window positions in 5.  (Indices run past
  // the last pixel to the end of its block's 32 to 256 pixels or of its grid row: those divide 2^31, so they fit where
  // `pixels` does.)
  const int64_t images = 63 / P + 2;
  const bool narrow = fitsInt(pixels) && fitsInt(images * IC * H * W * 4) && fitsInt(images * OC * P * 4) &&
                      fitsInt(65 * K * 4) && KH <= 31 && KW <= 31;
  // Few taps: stores written through to memory (us, not / written through: 12 x 1 x 12 x 91 -> 256 7.8 / 6.9, 8 x 3 x 224 x 224 ->
  // 64 of stride 2 16.1 / 14.4, 8 x 3 x 224 x 224 -> 64 33.2 / 31.8), unless much is written and a tile's runs of 32 pixels are no whole
  // lines, which then go to memory twice (4 x 3 x 223 x 225 -> 64, 51 MB, 20.1 / 20.6, 103 MB 40.9 / 47.1; 28 MB 10.3 / 9.1), and
  // not beside an addend, whose loads wait for them (6 x 1 x 12 x 91 -> 256 7.0 / 9.7).
  const bool through = P % 32 == 0 || N * OC * P * 4 <= int64_t(32) << 20;
  auto few = [&](auto octs, auto nss) {
    constexpr int OCT = decltype(octs)::value, NS = decltype(nss)::value;
    // two blocks per CU and channel tile at the registers of OCT = 2, four at those of OCT = 1
    const int64_t most = std::max<int64_t>(1, (int64_t)numComputeUnits() * (4 / OCT) / ((OC + 32 * OCT - 1) / (32 * OCT)));
    const int64_t blocks = std::min((pix32 + 3) / 4, most);
    auto *kernel = add ? conv_few_taps_kernel<OCT, NS, Output::Added>
                       : through ? conv_few_taps_kernel<OCT, NS, Output::Through> : conv_few_taps_kernel<OCT, NS, Output::Cached>;
    launchKernel(kernel, gridOf(blocks, 32 * OCT, 256), dim3(256), stream,
        input, weight, bias, output, g, (int)OC, (int)P, (int)N, byP, byOW, add, relu, (int)K, (int)pix32, (int)(4 * blocks));
  };
  const int64_t tiles128 = (pixels + 127) / 128;
  // Four pixels a lane: stores written through to memory, but (us, plain / written through / non-temporal, among passes on other inputs)
  //  * non-temporal where the output fills the Infinity Cache by itself: 16 x 3 x 256 x 256 -> 64, 256 MiB, 65 / 63 / 57, 35 x 8 x 256 x 256 -> 32
  //    76 / 72 / 56; of 135 MiB 30.9 / 26.7 / 31.3, and a pass that is waited for is slower so (216 MiB 49 / 46 / 55);
  //  * plain where much is written and a tile's runs are no whole lines, of which non-temporal stores write each piece on its own: 14 x 4 x 193 x
  //    188 -> 96, 186 MiB, 52 / 70 / 63, 17 x 1 x 101 x 68 -> 512 70 / 90 / 83; of 65 MiB 18.2 / 17.0 / 24.6, 86 18.1 / 17.0 / 27.2;
  //    (where nothing of the output is in that cache from the pass before, plain stores are ahead of both from some 32 MiB on, by 10 % at 100 MiB);
  //  * beside an addend non-temporal beyond 128 MiB (29 x 8 x 241 x 176 -> 32, 150 MiB, 73.6 / 71.1 / 68.3).
  const int64_t written = N * OC * P * 4, MiB = int64_t(1) << 20;
  const Output quadStores = add ? (written > 128 * MiB ? Output::Streamed : Output::Through)
                            : P % 32 ? (written > 128 * MiB ? Output::Cached : Output::Through)
                                     : written >= 256 * MiB ? Output::Streamed : Output::Through;
  auto quads = [&](auto kw, auto nr) {
    constexpr int KWC = decltype(kw)::value, NR = decltype(nr)::value;
    // two blocks per CU and channel tile
    const int64_t most = std::max<int64_t>(1, (int64_t)numComputeUnits() * 2 / ((OC + 31) / 32));
    const int64_t blocks = std::min((tiles128 + 3) / 4, most);
    // In pieces from 12 taps on (fewer leave half of the sixteen products of an instruction for nothing); an addend in flight leaves no
    // registers for them.
    auto kernelOf = [&](auto split) {
      constexpr bool SPLIT = decltype(split)::value;
      return quadStores == Output::Streamed ? conv_quads_kernel<KWC, NR, Output::Streamed, false, SPLIT>
             : quadStores == Output::Cached ? conv_quads_kernel<KWC, NR, Output::Cached, false, SPLIT> : conv_quads_kernel<KWC, NR, Output::Through, false, SPLIT>;
    };
    auto *kernel = kernelOf(std::false_type());
    if (add) kernel = quadStores == Output::Streamed ? conv_quads_kernel<KWC, NR, Output::Streamed, true, false> : conv_quads_kernel<KWC, NR, Output::Through, true, false>;
    else if constexpr (KWC * NR > 8)
      if (K >= 12) kernel = kernelOf(std::true_type());
    launchKernel(kernel, gridOf(blocks, 32, 256), dim3(256), stream, input, weight, bias, output, g, (int)OC, (int)P, (int)N, byP, byOW, add, relu,
                                                              (int)tiles128, (int)(4 * blocks));
  };
  const int64_t across = (OW + 31) / 32;
  auto patch = [&](auto kw, auto nr, auto sw) {
    constexpr int KWC = decltype(kw)::value, NR = decltype(nr)::value, SWC = decltype(sw)::value;
    const int64_t rowTiles = N * OH * across;
    // two blocks per CU and channel tile
    const int64_t most = std::max<int64_t>(1, (int64_t)numComputeUnits() * 2 / ((OC + 31) / 32));
    const int64_t blocks = std::min((rowTiles + 3) / 4, most);
    auto *kernel = add ? conv_patch_kernel<KWC, NR, SWC, true> : conv_patch_kernel<KWC, NR, SWC, false>;
    launchKernel(kernel, gridOf(blocks, 32, 256), dim3(256), stream, input, weight, bias, output, g, (int)OC, (int)P, (int)N, fastDiv((int)across),
                                                              byOH, add, relu, (int)across, (int)rowTiles, (int)(4 * blocks));
  };
  auto window = [&](auto win, auto pts, auto kss) {
    constexpr int WIN = decltype(win)::value, PT = decltype(pts)::value, KS = decltype(kss)::value;
    const int64_t perBlock = 4 / KS * 32 * PT;
    launchKernel(conv_window_kernel<WIN, PT, KS>, gridOf((pixels + perBlock - 1) / perBlock, 32, 256), dim3(256), stream,
        input, weight, bias, output, g, (int)OC, (int)P, (int)N, byP, byOW, add, relu);
  };
  auto staged = [&](auto win, auto kss) {
    constexpr int WIN = decltype(win)::value, KS = decltype(kss)::value;
    launchKernel(conv_staged_kernel<WIN, KS>, gridOf(pix32, 32, 64 * KS), dim3(64 * KS), stream,
        input, weight, bias, output, g, (int)OC, (int)P, (int)N, byP, byOW, add, relu);
  };
  auto tile = [&](auto win, auto kss) {
    constexpr int WIN = decltype(win)::value, KS = decltype(kss)::value;
    launchKernel(conv_tile_kernel<WIN, KS>, gridOf((pixels + 63) / 64, 64, 256 * KS), dim3(256 * KS), stream,
        input, weight, bias, output, g, (int)OC, (int)P, (int)N, byP, byOW, add, relu);
  };
  auto table = [&](auto wide) {
    launchKernel(conv_table_kernel<decltype(wide)::value>, gridOf(pix32, 32, 256), dim3(256), stream,
        input, weight, bias, add, output, g, (int)OC, (int)K, (int)P, pixels, relu);
  };
  using std::integral_constant;
  const integral_constant<int, 1> c1{};
  const integral_constant<int, 2> c2{};
  const integral_constant<int, 4> c4{};
  // A 32 x 32 tile per wavefront group: `tiles` of them.  Measured where the lines lie (us, the
  // kernels in turn, 3 x 3 unless said otherwise):
  //  * 196 tiles (4 x 64 x 28 x 28 -> 64): window x 4 wavefronts 7.0, LDS tiles 14.7-18; 136 tiles
  //    (256 x 13 x 41 -> 256): 18.0 against 45-62; 784 tiles (8 x 256 x 14 x 14 -> 512): 70 against 45;
  //  * LDS tiles: 200 blocks of 128 units 45.5 with four groups, 49.3 with two, 62.8 with one; 392 blocks
  //    of 32 units 29.9 / 25.9 / 27.9; 284 blocks of 16 units (1 x 1) 29.8 / 24.8 / 23.5;
  //  * 96 channels are two 64-channel tiles with a quarter of nothing: 12 x 32 x 100 x 90 -> 96 takes 87 in LDS
  //    tiles and 66-75 in window tiles of two accumulators.
  const int64_t tiles = pix32 * ((OC + 31) / 32);
  //    (Squares of 3, 5 and 7 come here only where convStagedWaves leaves them.)
  const bool squareWindow = KH == KW && (KH == 1 || KH == 3 || KH == 5 || KH == 7);
  if (!narrow) {
    table(std::true_type());
  } else if (K <= 32) {
    // Four pixels a lane from two tiles of 32 x 128 a CU on (us, pixel by pixel / quads, 3 x 3 from 3 channels: 256 tiles 5.2 / 6.9,
    // 512 6.9 / 7.2 and 6.8 / 6.4, 768 10.2 / 7.8, 1024 11.2 / 7.9, 2048 15.5 / 12.8); not from more than 16 window rows, whose
    // taps leave no registers to prefetch into (1 x 1 from 32 channels, 2048 tiles: 18.8 / 23.0).
    const int64_t rows = IC * KH;
    const bool wholeQuads = OW % 4 == 0 && OW <= W && SW == 1 && PWL < KW && (KW == 1 || ((KW == 3 || KW == 5) && DW == 1));
    if (wholeQuads && rows <= 16 && tiles128 * ((OC + 31) / 32) >= 2 * numComputeUnits() &&
        fitsInt((127 / P + 2) * IC * H * W * 4) && fitsInt((127 / P + 2) * OC * P * 4)) {
      if (KW == 1 && rows <= 4) quads(c1, c2);
      else if (KW == 1 && rows <= 8) quads(c1, c4);
      else if (KW == 1) quads(c1, integral_constant<int, 8>());
      else if (KW == 3 && rows <= 4) quads(integral_constant<int, 3>(), c2);
      else if (KW == 3 && rows <= 6) quads(integral_constant<int, 3>(), integral_constant<int, 3>());
      else if (KW == 3) quads(integral_constant<int, 3>(), integral_constant<int, 5>());
      else quads(integral_constant<int, 5>(), integral_constant<int, 3>());
      MGPU_CHECK_LAUNCH("mgpuConv2d");
      return;
    }
    auto steps = [&](auto octs) {
      if (K <= 10) few(octs, integral_constant<int, 5>());
      else if (K <= 16) few(octs, integral_constant<int, 8>());
      else if (K <= 28) few(octs, integral_constant<int, 14>());
      else few(octs, integral_constant<int, 16>());
    };
    // (two accumulators share the gathered taps; few pixels are spread over more wavefronts instead)
    if (OC > 32 && pix32 >= 4 * numComputeUnits()) steps(c2);
    else steps(c1);
  } else if (squareWindow && DW == 1 && fitsInt(N * OH * across) &&
             convByPatches((int)KH, (int)SW, tiles, N * OH * across * ((OC + 31) / 32), IC, OC, OW, numComputeUnits())) {
    auto go = [&](auto kw, auto nr) {
      if (SW == 1) patch(kw, nr, c1);
      else patch(kw, nr, c2);
    };
    if (KH == 5) go(integral_constant<int, 5>(), integral_constant<int, 8>());
    else if (IC == 1) go(integral_constant<int, 7>(), c4);
    else go(integral_constant<int, 7>(), integral_constant<int, 11>());
  } else if (squareWindow) {
    // 3 x 3 from 32 channels on in three bf16 numbers, where both estimates say that this is faster (700 shapes: taken by 267, 0.91 of the
    // time over all of them where the best choice everywhere would be 0.907, 0.66 beyond 80 us, two 5 to 6 % slower).  (16 channels are one
    // step: no gain.)
    ConvSplitPlan split{0, 0, 0.0};
    if (KH == 3 && IC >= 32 && IC % 16 == 0) {
      const int cus = numComputeUnits();
      split = convSplitPlan((int)N, (int)IC, (int)OC, (int)OH, (int)OW, (int)SH, (int)SW, (int)DH, (int)DW, cus, 0.97 * convWindowTime(SH, pixels, IC, OC, OW, cus));
    }
    // 5 x 5 and 7 x 7 from 16 channels on likewise.  What the other kernels take is estimated low, by the matrix instructions of the rounds alone
    // (5 x 5 0.131 to 0.25 us a round and channel were measured, 7 x 7 0.262 to 0.36; this leaves some launches of one or two rounds with them.
    // 500 shapes each: taken by 168 and 175, 0.886 and 0.908 of the time over all of them where the best choice would be 0.875 and 0.902, none
    // slower; an estimate a tenth higher, 0.881 and 0.905, is up to 10 % wrong).
    if (KH >= 5 && IC >= 16 && IC % (KH == 5 ? 8 : 4) == 0) {
      const int cus = numComputeUnits();
      const double others = 3.0 + (double)((tiles + cus - 1) / cus) * (KH == 5 ? 0.13 : 0.27) * (double)IC;
      split = (KH == 5 ? convSplitPlan5 : convSplitPlan7)((int)N, (int)IC, (int)OC, (int)OH, (int)OW, (int)SH, (int)SW, (int)DH, (int)DW, cus, others);
    }
    // Few tiles on quarters or halves of them, where the estimates say so by 8 % (570 launches of up to 1300 quarters: 0.81 of the time on
    // average, the best choice everywhere would be 0.80, three of them 3 to 6 % slower; by 5 % 20 of them would be, of 24 channels).
    if (KH >= 3) {
      const int cus = numComputeUnits();
      const double others = convFewTilesTime((int)KH, SH, pixels, IC, OC, OW, cus);
      const ConvSmallPlan small = convSmallPlan((int)KH, pixels, IC, OC, cus);
      if (small.ocSide && small.us < 0.92 * (split.strips ? std::min(others, 1.05 * split.us) : others) &&
          convSmall((int)KH, small.ocSide, input, weight, bias, output, add, N, IC, H, W, OC, OH, OW, PHL, PWL, SH, SW, DH, DW, relu, stream)) {
        MGPU_CHECK_LAUNCH("mgpuConv2d");
        return;
      }
    }
    if (split.strips && convSplit(split, input, weight, bias, output, add, N, IC, H, W, OC, OH, OW, PHL, PWL, SH, SW, DH, DW, relu, stream)) {
      MGPU_CHECK_LAUNCH("mgpuConv2d");
      return;
    }
    // (convWindowTime restates these lines for 3 x 3, and convFewTilesTime the first two: what changes here changes there.)
    auto pick = [&](auto win) {
      constexpr int WIN = decltype(win)::value;
      const int64_t units = ((IC + 2 * Window<WIN>::HALF - 1) / (2 * Window<WIN>::HALF)) * Window<WIN>::UNITS;
      const int64_t blocks = (pixels + 63) / 64 * ((OC + 63) / 64);
      if constexpr (WIN >= 3) {
        const int ks = convStagedWaves(WIN, SW, pixels, IC, OC, OW, numComputeUnits());
        if (ks == 8) return staged(win, integral_constant<int, 8>());
        if (ks == 4) return staged(win, c4);
      }
      if (tiles <= 400) window(win, c1, c4);
      else if ((OC - 1) % 64 >= 32) {
        if (blocks <= numComputeUnits() && units >= 64) tile(win, c4);
        else if (blocks <= 2 * numComputeUnits() && units >= 24) tile(win, c2);
        else tile(win, c1);
      } else if (tiles <= 2048) window(win, c1, c2);
      else if constexpr (WIN <= 3) window(win, c2, c1);
      else window(win, c1, c1);
    };
    if (KH == 1) pick(c1);
    else if (KH == 3) pick(integral_constant<int, 3>());
    else if (KH == 5) pick(integral_constant<int, 5>());
    else pick(integral_constant<int, 7>());
  } else {
    table(std::false_type());
  }
  MGPU_CHECK_LAUNCH("mgpuConv2d");
}

void pool2d(const float *input, float *output, int64_t N, int64_t C, int64_t H, int64_t W, int64_t OH, int64_t OW,
            int64_t KH, int64_t KW, int64_t PHL, int64_t PWL, int64_t PHR, int64_t PWR, int64_t SH, int64_t SW,
            int64_t method, hipStream_t stream) {
  if (N < 0 || C < 0 || H <= 0 || W <= 0 || OH < 0 || OW < 0 || KH <= 0 || KW <= 0) fail("mgpuPool2d: bad shape");
  if (PHL < 0 || PWL < 0 || PHR < 0 || PWR < 0 || SH <= 0 || SW <= 0) fail("mgpuPool2d: bad padding or stride");
  if (method != 0 && method != 1) fail("mgpuPool2d: method is 0 (max) or 1 (average)");
  const int64_t spanH = H + PHL + PHR - KH, spanW = W + PWL + PWR - KW;
  if (spanH < 0 || spanW < 0 || OH != spanH / SH + 1 || OW != spanW / SW + 1)
    fail("mgpuPool2d: output size does not follow from input, kernel, padding and stride");
  if (PHL >= KH || PWL >= KW || PHR >= KH || PWR >= KW) fail("mgpuPool2d: padding must be smaller than the window");
  if (N == 0 || C == 0) return;
  if (!input || !output) fail("mgpuPool2d: null pointer");
  for (int64_t v : {H, W, OH, OW, KH, KW, PHL, PWL, SH, SW})
    if (!fitsInt(v)) fail("mgpuPool2d: dimension too large");
  const int64_t total = N * C * OH * OW;
  const unsigned blocks = blocksFor(total);
  auto launch = [&](auto index) {
    using Index = decltype(index);
    launchKernel(pool_kernel<Index>, dim3(blocks), dim3(256), stream, input, output, (Index)total, (Index)blocks * 256, (int)H, (int)W, (int)OH,
                                                               (int)OW, (int)KH, (int)KW, (int)PHL, (int)PWL, (int)SH, (int)SW, method == 1);
  };
  // (the stride is added past the last index once)
  if (N * C * H * W <= 0x7fffffff && total + (int64_t)blocks * 256 <= 0xffffffffll) launch(uint32_t());
  else launch(int64_t());
  MGPU_CHECK_LAUNCH("pool_kernel");
}

} // namespace mgpu
