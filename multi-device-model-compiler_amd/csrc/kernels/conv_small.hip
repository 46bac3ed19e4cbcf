// Convolution of fp32 tensors with a 3 x 3, 5 x 5 or 7 x 7 window on tiles of 16 pixels x 16 output channels, for launches whose tiles of 32 x 32
// would leave most CUs idle: 64 pixels of a network's last stages are two or three such tiles, each a chain of thousands of products.
//
// v_mfma_f32_16x16x4_f32 does as many products a cycle as the 32 x 32 x 2 form of the other kernels, so a tile of a quarter has a
// quarter of the matrix instructions on four times as many CUs, and loses only in operands: a tap is loaded for 16 channels, a filter value
// for 16 pixels.  Where quarters would be two rounds of the CUs and halves one, a block takes 32 channels, which share the taps.
// A block's eight wavefronts split the input channels, four at a time (a lane quarter each); their sums meet in LDS.  Filter rows go
// through LDS along the rows, as in conv_staged_kernel, in an area of the wavefront's own (no barrier in the loop); a tap's byte offset is
// a register, the channel the scalar offset of the load.
//
// What bounds it: launch, first loads and the sum of the wavefronts' shares (3 to 4 us), then the L1, which takes about 8 cycles a tap
// load (a line or two for each channel of the four) and 16 a load of filter rows: 27 cycles a channel and 3 x 3 window, of which the matrix
// cores need 18.  us, before / now, 3 x 3: 2640 pixels of 256 -> 16 14.0 / 7.3, 510 of 256 -> 256 14.4 / 10.0, 540 of 128 -> 128 9.0 / 6.5; 5 x 5
// 1152 of 256 -> 64 33.1 / 22.7; 7 x 7 576 of 64 -> 64 19.7 / 9.0, 180 of 256 -> 8 69.6 / 29.9.  Error against 64 bits 0.6e-7 to 2.4e-7 where it
// was 0.6e-7 to 3.3e-7: a wavefront's sums are shorter and go in two chains.
#include "common.hpp"
#include "conv.hpp"
#include "mfma.hpp"
#include "mgpu_ops_internal.hpp"

#include <algorithm>

namespace mgpu {

namespace {

constexpr int kShares = 8; // wavefronts of a block
constexpr int kSide = 16;  // of a tile
constexpr int kGroup = 4;  // channels at a time

struct SmallGeo {
  int IC, H, W, OW, PHL, PWL, SH, SW, DH, DW;
  int blocks, inner; // tiles; those side by side that are counted first, of pixels where the filter is the larger operand, else of channels
  FastDiv byInner;
  bool pixelsFirst;
};

template <int WIN, int OT> struct Small {
  static constexpr int KK = WIN * WIN;
  static constexpr int UNITS = WIN == 3 ? 1 : WIN, STEPS = KK / UNITS; // taps fetched at a time: the window, or one of its rows
  static constexpr int CG = WIN == 3 ? 2 : 1;                          // groups staged at a time
  static constexpr int ROW = CG * kGroup * KK;                         // floats of a channel's row among them
  static constexpr int PITCH = ROW / 4 % 2 ? ROW : ROW + 4;            // 4 times an odd number of words: 16 rows and 4 quarters on 64 banks
  static constexpr int ROWS = OT * kSide, PIECES = ROW / 4, LOADS = (ROWS * PIECES + 63) / 64;
  static_assert(KK % 4 == 1, "a quarter's values one bank past the last's");
};

// OT: tiles of 16 channels beside each other
template <int WIN, int OT>
__global__ __launch_bounds__(64 * kShares, 2) void conv_small_kernel(const float *__restrict__ x, const float *__restrict__ w, int OC, int P, int N,
                                                                     FastDiv byP, FastDiv byOW, const float *__restrict__ bias,
                                                                     float *__restrict__ y, const float *__restrict__ add, int relu, SmallGeo g) {
  using S = Small<WIN, OT>;
  constexpr int KK = S::KK, UNITS = S::UNITS, STEPS = S::STEPS, kArea = S::ROWS * S::PITCH;
  static_assert(kArea >= S::ROWS * kSide && S::ROWS * kSide <= 64 * kShares, "the sums take the filter rows' place, and a thread finishes one");
  __shared__ __attribute__((aligned(16))) float smem[kShares * kArea];

  const int tid = threadIdx.x, lane = tid % 64;
  const int share = __builtin_amdgcn_readfirstlane(tid / 64);
  const int l16 = lane % 16, quarter = lane / 16;
  // An equal run of tiles for each XCD, those one after another that share the larger operand, which then comes into one L2 (168 pixels
  // of 256 -> 512, 7 x 7, 26 MB of filter: 90 us with every eighth tile on an XCD, 84 so; over 300 launches 0.97 of the time).
  const int xcd = (int)blockIdx.x % 8, run = g.blocks / 8, extra = g.blocks % 8;
  const int wid = xcd * run + (xcd < extra ? xcd : extra) + (int)blockIdx.x / 8;
  const int outer = __builtin_amdgcn_readfirstlane(divide(wid, g.byInner)), inner = wid - outer * g.inner;
  const int oc0 = (g.pixelsFirst ? outer : inner) * S::ROWS, q0 = (g.pixelsFirst ? inner : outer) * kSide;
  const int HW4 = g.H * g.W * 4, pixels = N * P;
  const int nFirst = __builtin_amdgcn_readfirstlane(divide(q0, byP));

  const int groups = g.IC / kGroup; // (whole: the launcher sees to it)
  const int g0 = groups * share / kShares, g1 = groups * (share + 1) / kShares;

  // Filter rows: piece p of 16 bytes is piece p % PIECES of channel p / PIECES.  (A channel past the end reads the last one's row and is
  // not stored; groups past the share are loaded and not used, past the row read as the next one's, past the filter as 0.)
  const auto filter = resource(w + (int64_t)oc0 * g.IC * KK, (int64_t)(OC - oc0) * g.IC * KK);
  float *mine = smem + share * kArea;
  int woff[S::LOADS];
#pragma unroll
  for (int i = 0; i < S::LOADS; i++) {
    const int p = i * 64 + lane, oc = p / S::PIECES;
    woff[i] = oc < S::ROWS ? ((oc0 + oc < OC ? oc : OC - 1 - oc0) * g.IC * KK + 4 * (p - oc * S::PIECES)) * 4 : kOutside;
  }
  u32x4 stage[S::LOADS];
  auto load = [&](int group) {
#pragma unroll
    for (int i = 0; i < S::LOADS; i++) stage[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(filter, woff[i], group * (kGroup * KK * 4), 0));
  };
  auto keep = [&]() {
#pragma unroll
    for (int i = 0; i < S::LOADS; i++) {
      const int p = i * 64 + lane, oc = p / S::PIECES;
      if (64 * (i + 1) <= S::ROWS * S::PIECES || oc < S::ROWS) *reinterpret_cast<u32x4 *>(mine + oc * S::PITCH + 4 * (p - oc * S::PIECES)) = stage[i];
    }
  };
  if (g0 < g1) load(g0); // (first of all, and what the end needs: the way to memory is most of a short launch)

  // The output that this thread finishes: channel and pixel tid of the tile, row by row.
  const int ocOut = oc0 + tid / kSide, qOut = q0 + tid % kSide;
  const bool finishes = tid < S::ROWS * kSide && ocOut < OC && qOut < pixels;
  int64_t outAt = 0;
  float bv = 0.0f, av = 0.0f;
  if (finishes) {
    const int n = divide(qOut, byP);
    outAt = ((int64_t)n * OC + ocOut) * P + (qOut - n * P);
    bv = bias[ocOut];
    if (add) av = add[outAt];
  }

  // A tap's byte offset, kOutside where it lies outside; 7 x 7, whose 49 would not leave the registers for the filter: the first window
  // row's, and in bit 31 - kh of rowOut which rows lie outside.
  int voff[WIN == 7 ? WIN : KK];
  unsigned rowOut = 0;
  {
    const int q = q0 + l16;
    const bool live = q < pixels;
    const int n = live ? divide(q, byP) : nFirst, p = live ? q - n * P : 0;
    const int oh = divide(p, byOW), ow = p - oh * g.OW;
    const int ih0 = live ? oh * g.SH - g.PHL : -0x3fff0000, iw0 = ow * g.SW - g.PWL;
    const int base = ((n - nFirst) * g.IC + quarter) * HW4 + ((oh * g.SH - g.PHL) * g.W + iw0) * 4;
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
  // The reduction walks units in a pipeline two deep: a unit's taps fly under the matrix instructions of the one before.
  auto fetch = [&](float (&b)[STEPS], int group, int unit) {
    const unsigned out = (rowOut << unit) & 0x80000000u;
    const int down = unit * g.DH * g.W * 4;
#pragma unroll
    for (int i = 0; i < STEPS; i++) {
      const int at = WIN == 7 ? (int)((unsigned)(voff[i] + down) | out) : voff[unit * STEPS + i];
      b[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(image, at, group * kGroup * HW4, 0));
    }
  };
  const float *ap = mine + l16 * S::PITCH + quarter * KK;
  f32x4 acc[OT][2]; // (two chains: a product need not wait for the one before it)
#pragma unroll
  for (int t = 0; t < OT; t++) acc[t][0] = acc[t][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto multiply = [&](const float (&b)[STEPS], int inChunk, int unit) {
#pragma unroll
    for (int i = 0; i < STEPS; i++)
#pragma unroll
      for (int t = 0; t < OT; t++)
        acc[t][i % 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(ap[t * (kSide * S::PITCH) + inChunk * (kGroup * KK) + unit * STEPS + i], b[i], acc[t][i % 2], 0, 0, 0);
  };
  constexpr int NU = S::CG * UNITS, TURN = NU % 2 ? 2 : 1; // units of a chunk; chunks until a unit's buffer is the first again
  float b[2][STEPS];
  if (g0 < g1) fetch(b[0], g0, 0);
  for (int turn = g0; turn < g1; turn += TURN * S::CG) {
#pragma unroll
    for (int h = 0; h < TURN; h++) {
      const int chunk = turn + h * S::CG;
      if (h && chunk >= g1) break; // (uniform)
      keep();
      if (chunk + S::CG < g1) load(chunk + S::CG);
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
  __syncthreads(); // the shares take the filter rows' place
  // accumulator register r of lane l: channel 4 (l / 16) + r, pixel l % 16
#pragma unroll
  for (int t = 0; t < OT; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) smem[share * (S::ROWS * kSide) + (t * kSide + 4 * quarter + r) * kSide + l16] = acc[t][0][r] + acc[t][1][r];
  __syncthreads();
  if (!finishes) return;
  float v = 0.0f;
#pragma unroll
  for (int s = 0; s < kShares; s++) v += smem[s * (S::ROWS * kSide) + tid];
  v += bv;
  if (add) v += av;
  // cuDNN's ReLU with CUDNN_NOT_PROPAGATE_NAN maps NaN to 0, as fmaxf does
  y[outAt] = relu ? fmaxf(v, 0.0f) : v;
}

} // namespace

// us: start + rounds of the CUs * 32 input channels (four for each wavefront) * a part for the window, fitted to 1100 launches of up to
// 1300 tiles (10th and 90th percentile 0.87 and 1.15 times what was measured; 7 x 7 0.83 and 1.24).
ConvSmallPlan convSmallPlan(int win, int64_t pixels, int64_t IC, int64_t OC, int64_t cus) {
  static const double time[2][3][2] = {{{3.95, 0.484}, {2.97, 1.70}, {1.9, 3.7}}, {{3.57, 0.796}, {2.86, 2.69}, {0.0, 0.0}}};
  ConvSmallPlan best{0, 0.0};
  if (IC % kGroup) return best;
  for (int i = 0; i < (win == 7 ? 1 : 2); i++) {
    const int64_t side = kSide << i, rounds = ((pixels + kSide - 1) / kSide * ((OC + side - 1) / side) + cus - 1) / cus;
    if (rounds > 2) continue; // (of which the fit knows too little: 4914 pixels of 64 -> 64 in three 10.2 -> 10.7 us)
    const double *t = time[i][(win - 3) / 2];
    const double us = t[0] + (double)(rounds * ((IC + kGroup * kShares - 1) / (kGroup * kShares))) * t[1];
    if (!best.ocSide || us < best.us) best = ConvSmallPlan{(int)side, us};
  }
  return best;
}

// Launches it; false where its indices would not fit.
bool convSmall(int win, int ocSide, const float *x, const float *w, const float *bias, float *y, const float *add, int64_t N, int64_t IC, int64_t H, int64_t W,
               int64_t OC, int64_t OH, int64_t OW, int64_t PHL, int64_t PWL, int64_t SH, int64_t SW, int64_t DH, int64_t DW, bool relu,
               hipStream_t stream) {
  auto fits = [](int64_t v) { return v >= 0 && v <= 0x7fffffff; };
  const int64_t P = OH * OW, pixels = N * P, tiles = (pixels + kSide - 1) / kSide, ocTiles = (OC + ocSide - 1) / ocSide;
  // byte offsets from a tile's first image and filter row on are 32 bits wide; a grid's threads are fewer than 2^32
  const int64_t images = (kSide - 2) / P + 2;
  if (IC % kGroup || !fits(pixels + kSide) || !fits(images * IC * H * W * 4) || !fits(ocSide * IC * win * win * 4) || tiles * ocTiles * (64 * kShares) >= (int64_t(1) << 32))
    return false;
  const bool pixelsFirst = OC * win * win > N * H * W;
  const int inner = (int)(pixelsFirst ? tiles : ocTiles);
  const SmallGeo g{(int)IC, (int)H, (int)W, (int)OW, (int)PHL, (int)PWL, (int)SH, (int)SW, (int)DH, (int)DW, (int)(tiles * ocTiles), inner, fastDiv(inner), pixelsFirst};
  auto *kernel = ocSide == 32 ? (win == 3 ? conv_small_kernel<3, 2> : conv_small_kernel<5, 2>)
                 : win == 3 ? conv_small_kernel<3, 1> : win == 5 ? conv_small_kernel<5, 1> : conv_small_kernel<7, 1>;
  launchKernel(kernel, dim3((unsigned)(tiles * ocTiles)), dim3(64 * kShares), stream, x, w, (int)OC, (int)P, (int)N, fastDiv((int)P), fastDiv((int)OW),
               bias, y, add, relu, g);
  return true;
}

} // namespace mgpu
