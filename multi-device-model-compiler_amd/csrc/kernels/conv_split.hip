// 3 x 3, 5 x 5 and 7 x 7 convolution of fp32 tensors on the bf16 matrix cores, with fp32's accuracy.
//
// Every operand is taken apart into three bf16 numbers, each the nearest to what those before it leave: all 24 bits, at fp32's range
// (the split of Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations", 2019).  Of the nine products of two such numbers six are summed up in fp32; the other three are at most 2^-23 of a
// product, whichever its size, 2^-26 in the root mean square, and of either sign.  The sums' errors, which are the larger ones, become
// fewer, since an instruction adds sixteen products at a time where the fp32 one adds two.  Relative error against 64 bits (2-norm;
// N(0, 1) pixels): 0.56e-7 to 2.0e-7 for 3 x 3, 0.54e-7 to 2.7e-7 for 5 x 5, 0.72e-7 to 3.2e-7 for 7 x 7, on average 0.82, 0.76 and 0.66 times
// that of the fp32 instructions on the same shapes and never more; of a product without others, which those round once, 0.94e-7 at
// most to 0.6e-7.  (Two fp16 numbers and a scale for a block, three products, took 0.75 of the time, and lost what is small beside the
// block's largest values: an input channel of 1e-6 of the others, weighted up again, was off by 2e-4.)
//
// Operands are multiplied by 2^24 first, so that the last piece of a number near fp32's smallest is no subnormal, and sums by 2^-48 at
// the end.  What becomes of infinities, NaNs and products beyond 2^80 is no finite sum; a block with one does its tile again with the
// fp32 instructions, which read the same LDS, for those sums only, so that no image's result depends on the images beside it.
//
// What bounds it: 6 x 32 cycles of a SIMD for 32 x 32 x 16 products where the fp32 instruction takes 8 x 64.  One block a CU: eight
// wavefronts (producers) bring operands into LDS, four (consumers) multiply, a step of sixteen input channels at a time,
// double-buffered.  A step of 32 x 256 takes 2.35 us, of which the matrix cores are busy 0.54 and the LDS 0.53 (0.4 of that bank conflicts);
// without conversions it would take 2.2, with half of the products 1.9.  (Eight producers, since a lone wavefront on a SIMD issues a vector
// instruction every eight cycles only.  Operands of a step's first set asked for ahead of the last one's products took 95 us for 84 on the
// first 7 x 7 below.)
//  * Filter rows come as they are, 576 bytes of a channel and step by one load into LDS, a step ahead, of which a lane takes
//    four channels of a position or more.  A producer converts the rows that it has loaded itself, so that they need neither a second buffer
//    nor a barrier.  (Straight into registers a load touched seven rows: 15 cycles an instruction.)
//  * Pixels: the input rows under the tile with their padding as zeros, so that a tap is one distance in LDS for all of them,
//    eight channels of a pixel a lane, in registers two steps ahead.  Rows of neighbouring images follow each other; wide images
//    are cut into strips of columns.
//  * In LDS both are eight channels in 16 bytes, the lane's operand of the matrix instruction.
// A consumer has 32 channels x 64 pixels; one, two or four of them share pixels and split the nine positions (tiles of 256, 128
// and 64 pixels).  us, fp32 instructions / this, 3 x 3 pad 1: 12 x 256 x 10 x 46 -> 256 83 / 46, 12 x 256 x 240 x 36 -> 16 151 / 95, 17 x 128 x
// 15 x 33 -> 128 45 / 27, 32 x 64 x 56 x 56 -> 64 75 / 69, 23 x 256 x 12 x 10 -> 256 37 / 31, 8 x 256 x 14 x 14 -> 512 46 / 31.
//
// 5 x 5 and 7 x 7: sixteen channels of their positions would not fit the LDS.  A step has eight or four, and a matrix
// instruction's sixteen products are two positions, one a lane half, or four, two side by side in a lane's sixteen bytes.  Positions past the
// window are fillers of zeros, filter and pixels.  (Positions' distances by the vector unit in place of scalars, and two positions of 7 x 7 that may
// lie in different rows, by four reads in place of two, were slower.)  us, fp32 instructions / this, stride 1: 5 x 5 8 x 128 x 21 x 42 -> 128 81 / 38, 16 x 64 x 46 x 46 ->
// 64 120 / 61, 8 x 32 x 60 x 60 -> 64 43 / 25.5, 4 x 256 x 30 x 30 -> 256 156 / 71; 7 x 7 16 x 64 x 30 x 44 -> 64 133 / 84, 9 x 32 x 50 x 56 -> 32 38 / 25, 2 x 128
// x 54 x 64 -> 128 133 / 79.
#include "common.hpp"
#include "conv.hpp"
#include "mfma.hpp"
#include "mgpu_ops_internal.hpp"

#include <algorithm>

namespace mgpu {

namespace {

constexpr int kConsumers = 4, kProducers = 8, kThreads = 64 * (kConsumers + kProducers);
constexpr int kOC = 32;                      // output channels of a block
constexpr int kPT = 2;                       // tiles of 32 pixels of a consumer

struct SplitGeo {
  int OH, OW, PHL, PWL, SH, SW, DH, DW;
  int strips, stripW; // columns of the output are cut into strips
  int pitch, rows;    // input columns of a strip, input rows of an image, with their padding
  int pixels;         // output pixels of all strips
  FastDiv byPixels, byStripW, byStrips, byPitch, byRows; // byPixels: OH * stripW
};

// A load from memory into LDS, 16 bytes a lane, of the first LANES lanes (see mfma.hpp; all lanes must be on around it).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <int LANES> __device__ __forceinline__ void ldsLoad16First(uint32_t offset, const char *base, uint32_t ldsAddr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(offset), "s"(base),
               "s"(ldsAddr), "s"(~0ull >> (64 - LANES))
               : "memory", "m0");
}
#pragma clang diagnostic pop

// WIN: the window; KS: consumers that share their pixels; CAP: staged pixels at most
template <int WIN, int KS_, int CAP_> struct SplitShape {
  static constexpr int TAPS = WIN * WIN, CH = WIN == 3 ? 16 : WIN == 5 ? 8 : 4; // positions; input channels of a step
  // Sixteen bytes hold eight channels of a position, or four of two.  A matrix instruction's set of sixteen products is two of them: a position
  // of sixteen channels, two of eight (the last one with a filler beside it), or four of four, two and two side by side in a window row, of which
  // the eighth is a filler.
  static constexpr int OCTETS = CH == 16 ? 2 : 1, CPS = CH < 8 ? CH : 8, BESIDE = 8 / CPS; // channels and positions in sixteen bytes
  static constexpr int PAIRED = 3 - OCTETS, UNITS = BESIDE == 2 ? WIN * 4 : TAPS, SETS = (UNITS + PAIRED - 1) / PAIRED;
  static constexpr int KS = KS_, CAP = CAP_, PXW = kConsumers / KS, PX = 32 * kPT * PXW;
  static constexpr int UNIT = OCTETS * kPieces * kOC * 16 + 80; // bytes of a unit's filter values (the 80: units side by side on different banks)
  static constexpr int HALF = OCTETS == 2 ? kPieces * kOC * 16 : UNIT; // from the values of a lane half to the other's
  static constexpr int FILTER = SETS * PAIRED * UNIT, PXB = 2 * CPS, PIXELS = OCTETS * kPieces * CAP * PXB; // PXB: bytes of a pixel's pieces
  static constexpr int ROW = CH * TAPS, PITCH = ROW + 4; // words of a channel's filter in a step
  static constexpr int RAW = kOC * PITCH * 4;
  static constexpr int LDS = 2 * (FILTER + PIXELS) + RAW;
  static constexpr int RPW = kOC / kProducers; // filter rows of a producer
  // Its lanes' share of them at a time: eight values, or four where eight would leave most lanes of the second time idle
  static constexpr int SHARE = OCTETS == 2 ? 4 : 8, ITEMS = RPW * OCTETS * UNITS * (8 / SHARE);
  static constexpr int WI = (ITEMS + 63) / 64, PI = (OCTETS * CAP + 64 * kProducers - 1) / (64 * kProducers);
  static_assert(CAP % 64 == 0 && ROW % 4 == 0 && ROW / 4 <= 64 && LDS + 1024 <= 160 * 1024, "whole wavefronts; a CU's LDS");
  static_assert(KS == 1 || kConsumers * kPT * 16 * 64 * 4 <= LDS, "the partial sums take the buffers' place");
};

template <int WIN, int KS, int CAP>
__global__ __launch_bounds__(kThreads) void conv_split_kernel(const float *__restrict__ w, const float *__restrict__ x, int IC, int OC,
                                                              int gridDimX, int ocTiles, FastDiv byOcTiles, int H, int W, int N, int relu,
                                                              const float *__restrict__ bias, float *__restrict__ y,
                                                              const float *__restrict__ add, SplitGeo g) {
  using S = SplitShape<WIN, KS, CAP>;
  constexpr int PXW = S::PXW, PI = S::PI, WI = S::WI, RPW = S::RPW, TAPS = S::TAPS, SETS = S::SETS, CPS = S::CPS, PXB = S::PXB, SHARE = S::SHARE;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[S::LDS];
  __shared__ int bad;
  __shared__ float biasOf[kOC];

  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const bool producer = wave >= kConsumers;
  const int l32 = lane % 32, hl = lane / 32;
  // an equal run of tiles for each XCD, channel tiles of the same pixels one after another
  const int nblk = (int)gridDimX, xcd = (int)blockIdx.x % 8, share = nblk / 8, extra = nblk % 8;
  const int wid = xcd * share + (xcd < extra ? xcd : extra) + (int)blockIdx.x / 8;
  const int pxTile = __builtin_amdgcn_readfirstlane(divide(wid, byOcTiles)), ocTile = __builtin_amdgcn_readfirstlane(wid - pxTile * ocTiles);
  const int oc0 = ocTile * kOC, p0 = pxTile * S::PX;
  const int steps = IC / S::CH;
  const int pwave = wave - kConsumers;

  // ---- the filter, as it is: a producer loads the rows that it converts.  (Past the last step it is loaded once more, and so are the
  // pixels: a load on one path only would have every path wait for all of them.)
  constexpr int rawFrom = 2 * (S::FILTER + S::PIXELS);
  const float *raw = reinterpret_cast<const float *>(smem + rawFrom) + pwave * RPW * S::PITCH;
  const uint32_t rawAt = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) unsigned char *)smem) + rawFrom;
  auto atMost = [&](int step) { return step < steps ? step : steps - 1; };
  auto loadFilter = [&](int step) {
    const char *from = reinterpret_cast<const char *>(w) + (int64_t)step * (S::ROW * 4);
#pragma unroll
    for (int i = 0; i < RPW; i++) {
      const int row = pwave * RPW + i, oc = oc0 + row < OC ? oc0 + row : OC - 1; // (a channel past the end is not stored)
      ldsLoad16First<S::ROW / 4>((uint32_t)lane * 16, from + (int64_t)oc * (IC * TAPS * 4), rawAt + row * (S::PITCH * 4));
    }
  };
  if (producer) loadFilter(0);

  struct Pixel {
    int image, row, col; // of a strip of an image; output row and column in it
  };
  auto pixelOf = [&](int q) {
    Pixel p;
    p.image = divide(q, g.byPixels);
    const int r = q - p.image * (g.OH * g.stripW);
    p.row = divide(r, g.byStripW);
    p.col = r - p.row * g.stripW;
    return p;
  };
  // Staged input rows: from the first one of the tile's first pixel to the last one of its last, over the images.
  const Pixel first = pixelOf(p0), last = pixelOf((p0 + S::PX < g.pixels ? p0 + S::PX : g.pixels) - 1);
  const int r0 = first.image * g.rows + first.row * g.SH;
  const int staged = (last.image * g.rows + last.row * g.SH + (WIN - 1) * g.DH - r0 + 1) * g.pitch;
  const int blocks = __builtin_amdgcn_readfirstlane((staged + 63) / 64), plane = blocks * 64; // ... in pieces of 64 pixels
  const int n0 = __builtin_amdgcn_readfirstlane(divide(first.image, g.byStrips));
  const int HW = H * W;
  unsigned char *const pixelBuf = smem + 2 * S::FILTER;
  if (tid < kOC) biasOf[tid] = bias[oc0 + tid < OC ? oc0 + tid : OC - 1];
  if (tid == 0) bad = 0;

  if (producer) {
    // What this wavefront converts: piece i of the pixels of 8 channels ...
    int xoff[PI], xlds[PI];
    const int perPlane = 65536 / blocks + 1;
    auto piece = [&](int i) { return i * kProducers + kProducers - 1 - pwave; }; // (the first wavefronts have more of the filter)
#pragma unroll
    for (int i = 0; i < PI; i++) {
      const int half = piece(i) * perPlane >> 16, px = (piece(i) - half * blocks) * 64 + lane; // half: of the step's channels
      const int r = divide(px, g.byPitch), c = px - r * g.pitch;
      const int vr = r0 + r, image = divide(vr, g.byRows), ih = vr - image * g.rows - g.PHL;
      const int n = divide(image, g.byStrips), iw = (image - n * g.strips) * g.stripW * g.SW + c - g.PWL;
      const bool in = half < S::OCTETS && px < staged && n < N && (unsigned)ih < (unsigned)H && (unsigned)iw < (unsigned)W;
      xoff[i] = in ? ((n - n0) * IC * HW + half * 8 * HW + ih * W + iw) * 4 : kOutside;
      xlds[i] = (half * kPieces * plane + px) * PXB;
    }
    // ... and of its filter rows
    int wraw[WI], wlds[WI];
    bool wused[WI], wlast[WI]; // wlast: its second position is a filler
#pragma unroll
    for (int i = 0; i < WI; i++) {
      const int e = i * 64 + lane, row = e / (S::ITEMS / RPW), r = e - row * (S::ITEMS / RPW);
      const int part = r / S::UNITS, unit = r - part * S::UNITS; // part: eight or four channels of the step's
      wused[i] = 64 * (i + 1) <= S::ITEMS || e < S::ITEMS;
      wraw[i] = wused[i] ? row * S::PITCH + part * (SHARE * TAPS) + (S::BESIDE == 2 ? unit / 4 * WIN + unit % 4 * 2 : unit) : 0;
      wlast[i] = S::BESIDE == 2 && unit % 4 == 3;
      wlds[i] = unit * S::UNIT + (pwave * RPW + row) * 16 + (SHARE == 8 ? part * (kPieces * kOC * 16) : part / 2 * (kPieces * kOC * 16) + part % 2 * 8);
    }
    const auto image = resource(x + (int64_t)n0 * IC * HW, (int64_t)(N - n0) * IC * HW);
    struct Pieces {
      float v[PI][CPS];
    };
    auto loadPixels = [&](Pieces &p, int step) {
      const int at = step * S::CH * HW * 4;
#pragma unroll
      for (int i = 0; i < PI; i++)
#pragma unroll
        for (int k = 0; k < CPS; k++) p.v[i][k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(image, xoff[i], at + k * HW * 4, 0));
    };
    // A step's operands in three pieces, or as they are.  Of eight channels as they are the first four go into one plane, the others
    // into the next; of two positions of four channels two each.
    auto put = [&](auto splitTag, const auto &v, unsigned char *at, int next, int quarter) {
      constexpr bool SPLIT = decltype(splitTag)::value;
      constexpr int COUNT = sizeof(v) / sizeof(float), PAIRS = COUNT / 2;
      if constexpr (SPLIT) {
        typedef uint32_t words __attribute__((ext_vector_type(PAIRS)));
        words p[kPieces];
#pragma unroll
        for (int k = 0; k < PAIRS; k++) {
          uint32_t piece[kPieces];
          splitTriple(v[2 * k] * kSplitScale, v[2 * k + 1] * kSplitScale, piece);
#pragma unroll
          for (int i = 0; i < kPieces; i++) p[i][k] = piece[i];
        }
#pragma unroll
        for (int i = 0; i < kPieces; i++) *reinterpret_cast<words *>(at + i * next) = p[i];
      } else if constexpr (COUNT == 8) {
        constexpr int FIRST = CPS / 2;
        *reinterpret_cast<f32x4 *>(at) = f32x4{v[0], v[1], v[FIRST == 4 ? 2 : 4], v[FIRST == 4 ? 3 : 5]};
        *reinterpret_cast<f32x4 *>(at + next) = f32x4{v[FIRST], v[FIRST + 1], v[6], v[7]};
      } else if constexpr (CPS == 8) { // (quarter: which four of the eight)
        *reinterpret_cast<f32x4 *>(at + (quarter ? next - 8 : 0)) = f32x4{v[0], v[1], v[2], v[3]};
      } else {
        *reinterpret_cast<f32x2 *>(at) = f32x2{v[0], v[1]};
        *reinterpret_cast<f32x2 *>(at + next) = f32x2{v[2], v[3]};
      }
    };
    auto produce = [&](auto splitTag) {
      Pieces even, odd;
      loadPixels(even, 0);
      loadPixels(odd, atMost(1));
      auto turn = [&](Pieces &p, int s) { // what step s reads
        if (s < steps) {
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PI * CPS) : "memory"); // the filter of step s has arrived
          float f[WI][SHARE];
#pragma unroll
          for (int i = 0; i < WI; i++)
#pragma unroll
            for (int k = 0; k < SHARE; k++) f[i][k] = raw[wraw[i] + k % CPS * TAPS + k / CPS];
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          loadFilter(atMost(s + 1));
          unsigned char *at = smem + (s & 1) * S::FILTER;
#pragma unroll
          for (int i = 0; i < WI; i++) {
#pragma unroll
            for (int k = CPS; k < SHARE; k++)
              if (wlast[i]) f[i][k] = 0.0f;
            if (wused[i]) put(splitTag, f[i], at + wlds[i], kOC * 16, wlds[i] & 8);
          }
          at = pixelBuf + (s & 1) * S::PIXELS;
#pragma unroll
          for (int i = 0; i < PI; i++)
            if (piece(i) < S::OCTETS * blocks) put(splitTag, p.v[i], at + xlds[i], plane * PXB, 0);
          loadPixels(p, atMost(s + 2));
        }
        __syncthreads();
      };
      turn(even, 0);
#pragma nounroll
      for (int s = 0; s < steps; s += 2) {
        turn(odd, s + 1);
        if (s + 1 < steps) turn(even, s + 2);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // (LDS gets another use)
    };
    produce(std::true_type());
    __syncthreads();
    if (bad) {
      loadFilter(0);
      produce(std::false_type());
    }
    if (KS > 1) __syncthreads();
    return;
  }

  // ---- consumers
  __builtin_amdgcn_s_setprio(3); // (theirs is the longer chain: 34.5 -> 32.7 us at 8 x 256 x 14 x 14 -> 512 in tiles of 256)
  const int ks = wave / PXW, pw = wave % PXW;
  int bbase[kPT], pix[kPT], img[kPT]; // the lane's pixels: in LDS, in their image (-1: none), and that
#pragma unroll
  for (int t = 0; t < kPT; t++) {
    const int q = p0 + (pw * kPT + t) * 32 + l32;
    const Pixel p = pixelOf(q < g.pixels ? q : p0);
    const int n = divide(p.image, g.byStrips), col = (p.image - n * g.strips) * g.stripW + p.col;
    bbase[t] = ((p.image * g.rows + p.row * g.SH - r0) * g.pitch + p.col * g.SW) * PXB + (S::OCTETS == 2 ? hl * (kPieces * 16) * plane : 0);
    pix[t] = q < g.pixels && col < g.OW ? p.row * g.OW + col : -1;
    img[t] = n - n0;
  }
  // The filler unit's filter values are zeros, which are taken for its pixels too (an infinity times 0 would be none).
  constexpr bool FILLED = S::UNITS % S::PAIRED != 0;
  constexpr int kFiller = S::UNITS * S::UNIT;
  if constexpr (FILLED) {
    constexpr int kEach = kPieces * kOC; // of sixteen bytes
    if (tid < 2 * kEach) *reinterpret_cast<u32x4 *>(smem + tid / kEach * S::FILTER + kFiller + tid % kEach * 16) = u32x4{0u, 0u, 0u, 0u};
  }
  f32x16 acc[kPT];
  auto multiply = [&](auto splitTag, f32x16 (&sum)[kPT]) {
    constexpr bool SPLIT = decltype(splitTag)::value;
    constexpr int PLANES = SPLIT ? kPieces : 2;
    f32x16 low[kPT]; // products with a lower piece: their roundings do not count among the others' (not SPLIT: every other product)
#pragma unroll
    for (int t = 0; t < kPT; t++)
#pragma unroll
      for (int i = 0; i < 16; i++) sum[t][i] = low[t][i] = 0.0f;
    struct Operands {
      bf16x8 a[PLANES], b[kPT][PLANES]; // not SPLIT: eight channels as two times four floats
    };
    auto read = [&](Operands &o, int step, int set) {
      const unsigned char *wat = smem + (step & 1) * S::FILTER + hl * S::HALF + l32 * 16 + set * (S::PAIRED * S::UNIT);
      const int pixelsAt = 2 * S::FILTER + (step & 1) * S::PIXELS;
      // (by scalars, and a selection between the lane halves)
      auto distance = [&](int unit) {
        const int ky = S::BESIDE == 2 ? unit / 4 : unit / WIN, kx = S::BESIDE == 2 ? unit % 4 * 2 : unit - ky * WIN;
        return (ky * g.DH * g.pitch + kx * g.DW) * PXB;
      };
      const int off = S::PAIRED == 2 && hl ? distance(2 * set + 1) : distance(S::PAIRED * set);
      const bool filler = FILLED && hl && set == SETS - 1;
#pragma unroll
      for (int i = 0; i < PLANES; i++) o.a[i] = *reinterpret_cast<const bf16x8 *>(wat + i * (kOC * 16));
#pragma unroll
      for (int t = 0; t < kPT; t++) {
        const int at = filler ? kFiller : pixelsAt + bbase[t] + off, next = filler ? 0 : plane * PXB;
#pragma unroll
        for (int i = 0; i < PLANES; i++) {
          if constexpr (S::BESIDE == 1) {
            o.b[t][i] = *reinterpret_cast<const bf16x8 *>(smem + at + i * next);
          } else { // (eight bytes of either pixel; behind the last one of a row lies what is none of the window's)
            const bf16x4 none = {}, *h = reinterpret_cast<const bf16x4 *>(smem + at + i * next);
            bf16x4 second = h[1];
            if (hl && set % 2) second = none;
            o.b[t][i] = __builtin_shufflevector(h[0], second, 0, 1, 2, 3, 4, 5, 6, 7);
          }
        }
      }
    };
    auto mma = [&](const Operands &o) {
      if constexpr (SPLIT) { // (the smallest products first)
        auto product = [&](f32x16 (&to)[kPT], int i, int k) {
#pragma unroll
          for (int t = 0; t < kPT; t++) to[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(o.a[i], o.b[t][k], to[t], 0, 0, 0);
        };
        product(low, 2, 0);
        product(low, 0, 2);
        product(low, 1, 1);
        product(sum, 0, 0);
        product(low, 1, 0);
        product(low, 0, 1);
      } else {
        // (a step of two products has one of either lane half: channel k and channel 8 + k)
#pragma unroll
        for (int k = 0; k < 8; k++) {
          const float a = __builtin_bit_cast(f32x4, o.a[k / 4])[k % 4];
#pragma unroll
          for (int t = 0; t < kPT; t++)
            (k % 2 ? low : sum)[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, __builtin_bit_cast(f32x4, o.b[t][k / 4])[k % 4], (k % 2 ? low : sum)[t], 0, 0, 0);
        }
      }
    };
    __syncthreads();
    for (int s = 0; s < steps; s++) {
      // sets from, from + KS, ...: dealt out in turns
      const int from = KS == 1 ? 0 : (ks + s * (SETS % KS)) % KS;
      Operands even, odd;
      read(even, s, from);
      int set = from;
#pragma nounroll
      for (; set + KS < SETS; set += 2 * KS) {
        read(odd, s, set + KS);
        // (5 x 5: reads first, where the compiler would save their registers and have every second set wait: 73 -> 70 us at 4 x 256 x 30 x
        // 30 -> 256.  3 x 3 gains nothing by it, 7 x 7 spills.)
        if (WIN == 5) __builtin_amdgcn_sched_barrier(0);
        mma(even);
        read(even, s, set + 2 * KS < SETS ? set + 2 * KS : from);
        if (WIN == 5) __builtin_amdgcn_sched_barrier(0);
        mma(odd);
      }
      if (set < SETS) mma(even);
      __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < kPT; t++) sum[t] += low[t];
  };
  multiply(std::true_type(), acc);
  bool finite = true;
#pragma unroll
  for (int t = 0; t < kPT; t++)
#pragma unroll
    for (int i = 0; i < 16; i++) finite = finite && fabsf(acc[t][i]) < __builtin_inff();
  if (!finite) bad = 1;
#pragma unroll
  for (int t = 0; t < kPT; t++) acc[t] *= kSplitUnscale;
  __syncthreads();
  if (bad) {
    f32x16 plain[kPT];
    multiply(std::false_type(), plain);
#pragma unroll
    for (int t = 0; t < kPT; t++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[t][i] = fabsf(acc[t][i]) < __builtin_inff() ? acc[t][i] : plain[t][i];
  }

  const int P = g.OH * g.OW;
  const int64_t outElems = (int64_t)OC * P;
  const auto out = resource(y + n0 * outElems, (N - n0) * outElems);
  const bool whole = oc0 + kOC <= OC; // (uniform)
  // accumulator register r of lane l: channel 8*(r/4) + 4*(l/32) + r%4, pixel l%32.  t: uniform
  auto finish = [&](int t, int r4, f32x4 v) { // registers r4 .. r4 + 3
    const int oc = 2 * r4; // less the lane's 4 hl
    const int pixel = t ? pix[1] : pix[0], at = pixel < 0 ? kOutside : (((t ? img[1] : img[0]) * OC + oc0 + 4 * hl) * P + pixel) * 4;
    int voff[4], soff[4];
    float a[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      soff[k] = whole || oc0 + oc + k < OC ? (oc + k) * P * 4 : 0; // (a scalar offset past the resource would wrap the check)
      voff[k] = whole || oc0 + oc + k + 4 * hl < OC ? at : kOutside;
      a[k] = 0.0f;
    }
    if (add) {
      const auto from = resource(add + n0 * outElems, (N - n0) * outElems);
#pragma unroll
      for (int k = 0; k < 4; k++) a[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(from, voff[k], soff[k], 0));
    }
    const f32x4 b = *reinterpret_cast<const f32x4 *>(&biasOf[oc + 4 * hl]);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const float r = v[k] + b[k] + a[k];
      // cuDNN's ReLU with CUDNN_NOT_PROPAGATE_NAN maps NaN to 0, as fmaxf does
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, relu ? fmaxf(r, 0.0f) : r), out, voff[k], soff[k], 0);
    }
  };
  if constexpr (KS == 1) {
#pragma unroll
    for (int t = 0; t < kPT; t++)
#pragma unroll
      for (int i = 0; i < 16; i += 4) finish(t, i, f32x4{acc[t][i], acc[t][i + 1], acc[t][i + 2], acc[t][i + 3]});
  } else { // the sum over the consumers of the same pixels, of which each finishes a share
    constexpr int QUADS = kPT * 4, SHARE = QUADS / KS;
    f32x4 *partial = reinterpret_cast<f32x4 *>(smem);
#pragma unroll
    for (int t = 0; t < kPT; t++)
#pragma unroll
      for (int i = 0; i < 16; i += 4)
        partial[(wave * QUADS + t * 4 + i / 4) * 64 + lane] = f32x4{acc[t][i], acc[t][i + 1], acc[t][i + 2], acc[t][i + 3]};
    __syncthreads();
#pragma unroll
    for (int i = 0; i < SHARE; i++) {
      const int q = ks * SHARE + i; // (uniform)
      f32x4 v = partial[(pw * QUADS + q) * 64 + lane];
#pragma unroll
      for (int s = 1; s < KS; s++) v += partial[((s * PXW + pw) * QUADS + q) * 64 + lane];
      finish(q / 4, q % 4 * 4, v);
    }
  }
}

// The tiles, and what a launch in them takes: us = start + rounds of the CUs * (block + step * steps), fitted to 580 to 700 launches of each
// of 3 x 3 and 410 to 500 of the others (a tenth to a ninetieth percentile of 0.91 to 1.04 times what was measured).
struct SplitTile {
  int pixels, cap;
  double start, block, step;
};
constexpr SplitTile kTiles[] = {{64, 256, 1.1, 3.8, 1.24}, {64, 448, 1.3, 4.2, 1.38}, {128, 256, 0.6, 5.0, 1.55}, {128, 448, 1.0, 5.1, 1.64}, {256, 448, 0.0, 7.2, 2.35},
                                {64, 512, 0.9, 3.85, 1.51}, {128, 512, 0.3, 5.1, 1.85}, {64, 960, 1.2, 3.9, 1.69}, {128, 960, 0.6, 4.85, 2.40}};
constexpr int kTiles3 = 5, kTiles5 = 2, kTiles7 = 2; // of 3 x 3, and behind them of 5 x 5 and 7 x 7

// The cheapest of tiles first .. first + count - 1, if it takes less than `limit` us.
ConvSplitPlan cheapest(int first, int count, int win, int step, int N, int IC, int OC, int OH, int OW, int SH, int SW, int DH, int DW, int cus, double limit) {
  ConvSplitPlan best{0, 0, limit};
  const int ocTiles = (OC + kOC - 1) / kOC, below = (win - 1) * DH + 1; // below: rows of a window
  for (int i = first; i < first + count; i++) {
    const SplitTile &tile = kTiles[i];
    const double round = tile.block + tile.step * (IC / step);
    if (tile.start + round >= best.us) continue;
    // the widest strips whose staged rows fit (none narrower than 8 beside others: their halo would be most of them)
    for (int strips = (OW + tile.cap - 1) / tile.cap, width; width = (OW + strips - 1) / strips, strips == 1 || width >= 8;
         strips = (OW + width - 2) / (width - 1)) {
      // rows that the tile's pixels lie in at most, and images; where one of these ends, its last window's rows come besides
      const int64_t rows = std::min<int64_t>((tile.pixels - 2) / width + 2, (int64_t)N * strips * OH);
      const int64_t images = std::min<int64_t>((tile.pixels - 2) / ((int64_t)OH * width) + 2, rows);
      const int64_t staged = ((rows - 1) * SH + below + (images - 1) * std::max(0, below - SH)) * ((int64_t)(width - 1) * SW + (win - 1) * DW + 1);
      if (staged <= tile.cap) {
        const int64_t blocks = ((int64_t)N * strips * OH * width + tile.pixels - 1) / tile.pixels * ocTiles;
        const double us = tile.start + (double)((blocks + cus - 1) / cus) * round;
        if (us < best.us) best = ConvSplitPlan{i, strips, us};
        break;
      }
      if (width == 1) break;
    }
  }
  return best;
}

} // namespace

ConvSplitPlan convSplitPlan(int N, int IC, int OC, int OH, int OW, int SH, int SW, int DH, int DW, int cus, double limit) {
  return cheapest(0, kTiles3, 3, 16, N, IC, OC, OH, OW, SH, SW, DH, DW, cus, limit);
}
ConvSplitPlan convSplitPlan5(int N, int IC, int OC, int OH, int OW, int SH, int SW, int DH, int DW, int cus, double limit) {
  return cheapest(kTiles3, kTiles5, 5, 8, N, IC, OC, OH, OW, SH, SW, DH, DW, cus, limit);
}
ConvSplitPlan convSplitPlan7(int N, int IC, int OC, int OH, int OW, int SH, int SW, int DH, int DW, int cus, double limit) {
  if (DW != 1) return ConvSplitPlan{0, 0, limit}; // (two positions of a row come as sixteen bytes side by side)
  return cheapest(kTiles3 + kTiles5, kTiles7, 7, 4, N, IC, OC, OH, OW, SH, SW, DH, DW, cus, limit);
}

// Launches it; false where its indices would not fit.
bool convSplit(const ConvSplitPlan &plan, const float *x, const float *w, const float *bias, float *y, const float *add, int64_t N, int64_t IC,
               int64_t H, int64_t W, int64_t OC, int64_t OH, int64_t OW, int64_t PHL, int64_t PWL, int64_t SH, int64_t SW, int64_t DH,
               int64_t DW, bool relu, hipStream_t stream) {
  auto fits = [](int64_t v) { return v >= 0 && v <= 0x7fffffff; };
  const int64_t strips = plan.strips, width = (OW + strips - 1) / strips, pixels = N * strips * OH * width, tilePixels = kTiles[plan.tile].pixels;
  const int win = plan.tile < kTiles3 ? 3 : plan.tile < kTiles3 + kTiles5 ? 5 : 7, taps = win * win;
  const int64_t pitch = (width - 1) * SW + (win - 1) * DW + 1, rows = (OH - 1) * SH + (win - 1) * DH + 1;
  const int64_t pxTiles = (pixels + tilePixels - 1) / tilePixels, ocTiles = (OC + kOC - 1) / kOC, blocks = pxTiles * ocTiles;
  // pixel, row and byte indices from a tile's first image on are 32 bits wide, the filter's from a channel on; a grid's threads are fewer than 2^32
  const int64_t images = (tilePixels - 2) / (OH * width) + 2;
  if ((win == 7 && DW != 1) || !aligned16(w) || !fits(pixels + tilePixels) || !fits(N * strips * rows + tilePixels * SH) || !fits(images * IC * H * W * 4) ||
      !fits(images * OC * OH * OW * 4) || !fits(IC * taps * 4) || blocks * kThreads >= (int64_t(1) << 32))
    return false;
  const SplitGeo g{(int)OH,    (int)OW, (int)PHL, (int)PWL,   (int)SH, (int)SW, (int)DH, (int)DW, (int)strips, (int)width, (int)pitch, (int)rows, (int)pixels,
                   fastDiv((int)(OH * width)), fastDiv((int)width), fastDiv((int)strips), fastDiv((int)pitch), fastDiv((int)rows)};
  auto launch = [&](auto *kernel) {
    launchKernel(kernel, dim3((unsigned)blocks), dim3(kThreads), stream, w, x, (int)IC, (int)OC, (int)blocks, (int)ocTiles, fastDiv((int)ocTiles), (int)H, (int)W,
                                                                  (int)N, relu, bias, y, add, g);
  };
  switch (plan.tile) {
  case 0: launch(conv_split_kernel<3, 4, 256>); break;
  case 1: launch(conv_split_kernel<3, 4, 448>); break;
  case 2: launch(conv_split_kernel<3, 2, 256>); break;
  case 3: launch(conv_split_kernel<3, 2, 448>); break;
  case 4: launch(conv_split_kernel<3, 1, 448>); break;
  case 5: launch(conv_split_kernel<5, 4, 512>); break;
  case 6: launch(conv_split_kernel<5, 2, 512>); break;
  case 7: launch(conv_split_kernel<7, 4, 960>); break;
  default: launch(conv_split_kernel<7, 2, 960>);
  }
  return true;
}

} // namespace mgpu
