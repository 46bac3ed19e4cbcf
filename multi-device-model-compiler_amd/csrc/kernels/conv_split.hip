// 3 x 3, 5 x 5 and 7 x 7 convolution of fp32 tensors on the fp16 matrix cores, with fp32's accuracy.
//
// Every operand is taken apart into two fp16 numbers, v = scale * x = hi + lo with hi = fp16(v), lo = fp16(v - hi) and a scale
// that is a power of two: 22 bits of the 24, and three products, hi.hi + (hi.lo + lo.hi), sum up in fp32.  What is left out is
// 2^-24 of a product, a rounding error of its own in every one; the sums' errors, which are the larger ones, become fewer, since
// an instruction adds sixteen products at a time where the fp32 one adds two.  Relative error against 64 bits (2-norm; N(0, 1)
// pixels, K taps): 0.9e-7 to 2.2e-7 for K = 288 to 2304, 1.2e-7 to 5.7e-7 with the fp32 instructions on the same shapes.
//
// What fp32 has and fp16 pairs have not is range.  The scales come from the block's own operands - one for its pixels, one for each
// output channel's filter, each from the largest value in its first step of input channels, which they put to 2^7 .. 2^8 -, so
// that tensors of any size fit, and the block checks while it converts: a value beyond 65504 (infinities; 256 times what the
// first channels hold), or a window whose largest value is under 2^-9 of them, and the block does its tile again with the fp32
// instructions, which read the same LDS.  (NaNs need no check: they come through both ways.)
//
// What bounds it: 3 x 32 cycles of a SIMD for 32 x 32 x 16 products where the fp32 instruction takes 8 x 64, so that moving and
// converting the operands is most of the work.  One block a CU: eight wavefronts (producers) bring operands into LDS, four
// (consumers) multiply, a step of sixteen input channels at a time, double-buffered.  (Eight producers, since a lone wavefront on
// a SIMD issues a vector instruction every eight cycles only: four took 2.1 us a step of 32 x 256, eight 1.5.)
//  * Filter rows come as they are, 576 bytes of a channel and step by one load into LDS, two steps ahead; a lane takes the eight
//    channels of one position from there.  (Straight into registers a load touched seven rows: 15 cycles an instruction.)
//  * Pixels: the input rows under the tile with their padding as zeros, so that a tap is one distance in LDS for all of them,
//    eight channels of a pixel a lane, in registers two steps ahead.  Rows of neighbouring images follow each other; wide images
//    are cut into strips of columns.
//  * In LDS both are eight channels in 16 bytes, the lane's operand of the matrix instruction.
// A consumer has 32 channels x 64 pixels; one, two or four of them share pixels and split the nine positions (tiles of 256, 128
// and 64 pixels).  us, before / now, 3 x 3 pad 1: 12 x 256 x 10 x 46 -> 256 83 / 34, 12 x 256 x 240 x 36 -> 16 151 / 67, 17 x 128 x
// 15 x 33 -> 128 46 / 20, 32 x 64 x 56 x 56 -> 64 77 / 53, 23 x 256 x 12 x 10 -> 256 40 / 25, 5 x 256 x 36 x 9 -> 256 26 / 21.
//
// 5 x 5 and 7 x 7: sixteen channels of their positions, twice and as they are, would not fit the LDS.  A step has eight or four, and a matrix
// instruction's sixteen products are two positions, one a lane half, or four, two side by side in a lane's sixteen bytes.  Positions past the
// window are fillers of zeros, filter and pixels.  The consumers' reads set the pace (1.5 us a step of 128 pixels, of which the matrix
// instructions are 0.5; three sets of operands on their way in place of two spill; positions' distances by the vector unit in place of
// scalars took 5 x 5 1.7 us, two positions of 7 x 7 that may lie in different rows, by four reads in place of two, 2.4).  us, before / now, stride 1:
// 5 x 5 8 x 128 x 21 x 42 -> 128 81 / 30, 16 x 64 x 46 x 46 -> 64 120 / 51, 8 x 32 x 60 x 60 -> 64 43 / 24, 4 x 256 x 30 x 30 -> 256 156 / 55; 7 x 7,
// tiles of 32 x 32, 1296 from 64 channels 140 / 61, 819 from 32 41 / 20, 432 from 128 70 / 46, 545 from 16 19.4 / 12.8.  Error against 64 bits 0.7e-7 to 1.6e-7
// for K = 400 to 3200, 0.8e-7 to 2.1e-7 before; 7 x 7 0.9e-7 to 2.3e-7, 1.3e-7 to 3.4e-7 before.
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
constexpr int kTop = 8;                      // scaled maxima lie under 2^8
constexpr float kMost = 65504.0f, kLeast = 0.25f; // what a pair holds; from where on to 2^-23

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

// The exponent of a scale 2^e for values whose largest has these bits (none: what to take them for where there is none).
__device__ __forceinline__ int scaleExponent(uint32_t largest, int none) {
  const int e = (int)(largest >> 23) - 126; // 2^(e-1) <= largest < 2^e
  return kTop - (largest == 0 || largest >= 0x7f800000u ? none : e < -100 ? -100 : e > 100 ? 100 : e);
}
__device__ __forceinline__ float powerOf2(int e) { return __builtin_bit_cast(float, (uint32_t)(e + 127) << 23); }

// WIN: the window; KS: consumers that share their pixels; CAP: staged pixels at most
template <int WIN, int KS_, int CAP_> struct SplitShape {
  static constexpr int TAPS = WIN * WIN, CH = WIN == 3 ? 16 : WIN == 5 ? 8 : 4; // positions; input channels of a step
  // Sixteen bytes hold eight channels of a position, or four of two.  A matrix instruction's set of sixteen products is two of them: a position
  // of sixteen channels, two of eight (the last one with a filler beside it), or four of four, two and two side by side in a window row, of which
  // the eighth is a filler.
  static constexpr int OCTETS = CH == 16 ? 2 : 1, CPS = CH < 8 ? CH : 8, BESIDE = 8 / CPS; // channels and positions in sixteen bytes
  static constexpr int PAIRED = 3 - OCTETS, UNITS = BESIDE == 2 ? WIN * 4 : TAPS, SETS = (UNITS + PAIRED - 1) / PAIRED;
  static constexpr int KS = KS_, CAP = CAP_, PXW = kConsumers / KS, PX = 32 * kPT * PXW;
  static constexpr int UNIT = OCTETS * 2 * kOC * 16 + 80; // bytes of a unit's filter values (the 80: units side by side on different banks)
  static constexpr int HALF = OCTETS == 2 ? 2 * kOC * 16 : UNIT; // from the values of a lane half to the other's
  static constexpr int FILTER = SETS * PAIRED * UNIT, PXB = 2 * CPS, PIXELS = OCTETS * 2 * CAP * PXB; // PXB: bytes of a pixel's pieces
  static constexpr int ROW = CH * TAPS, PITCH = ROW + 4; // words of a channel's filter in a step
  static constexpr int RAW = kOC * PITCH * 4, RAWS = 3;
  static constexpr int LDS = 2 * (FILTER + PIXELS) + RAWS * RAW;
  static constexpr int RPW = kOC / kProducers; // filter rows a producer moves
  static constexpr int ITEMS = kOC * OCTETS * UNITS; // sixteen bytes of a filter
  static constexpr int WI = (ITEMS + 64 * kProducers - 1) / (64 * kProducers), PI = (OCTETS * CAP + 64 * kProducers - 1) / (64 * kProducers);
  static_assert(CAP % 64 == 0 && ROW % 4 == 0 && ROW / 4 <= 64 && LDS + 1024 <= 160 * 1024, "whole wavefronts; a CU's LDS");
  static_assert(KS == 1 || kConsumers * kPT * 16 * 64 * 4 <= LDS, "the partial sums take the buffers' place");
};

template <int WIN, int KS, int CAP>
__global__ __launch_bounds__(kThreads) void conv_split_kernel(const float *__restrict__ w, const float *__restrict__ x, int IC, int OC,
                                                              int gridDimX, int ocTiles, FastDiv byOcTiles, int H, int W, int N, int relu,
                                                              const float *__restrict__ bias, float *__restrict__ y,
                                                              const float *__restrict__ add, SplitGeo g) {
  using S = SplitShape<WIN, KS, CAP>;
  constexpr int PXW = S::PXW, PI = S::PI, WI = S::WI, RPW = S::RPW, TAPS = S::TAPS, SETS = S::SETS, CPS = S::CPS, PXB = S::PXB;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[S::LDS];
  __shared__ uint32_t wMax[kOC], xMax;
  __shared__ int wExp[kOC], bad, small;
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
  const int pwave = wave - kConsumers, ptid = tid - 64 * kConsumers;

  // ---- the filter, as it is, into a ring of three steps.  (Past the last step it is loaded once more, and so are the pixels: a load
  // on one path only would have every path wait for all of them.)
  constexpr int rawFrom = 2 * (S::FILTER + S::PIXELS);
  const float *raw = reinterpret_cast<const float *>(smem + rawFrom);
  const uint32_t rawAt = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) unsigned char *)smem) + rawFrom;
  auto atMost = [&](int step) { return step < steps ? step : steps - 1; };
  auto loadFilter = [&](int step, int slot) {
    const char *from = reinterpret_cast<const char *>(w) + (int64_t)step * (S::ROW * 4);
#pragma unroll
    for (int i = 0; i < RPW; i++) {
      const int row = pwave * RPW + i, oc = oc0 + row < OC ? oc0 + row : OC - 1; // (a channel past the end is not stored)
      ldsLoad16First<S::ROW / 4>((uint32_t)lane * 16, from + (int64_t)oc * (IC * TAPS * 4), rawAt + slot * S::RAW + row * (S::PITCH * 4));
    }
  };
  if (producer) {
    loadFilter(0, 0);
    loadFilter(atMost(1), 1);
  }

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
  if (tid == 0) xMax = 0, bad = 0, small = 0;

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
      xlds[i] = (half * 2 * plane + px) * PXB;
    }
    // ... and sixteen bytes of the filter
    int wraw[WI], wlds[WI], wch[WI];
    bool wused[WI], wlast[WI]; // wlast: its second position is a filler
#pragma unroll
    for (int i = 0; i < WI; i++) {
      const int at = i * 64 * kProducers + ptid, e = at < S::ITEMS ? at : S::ITEMS - 1; // (past the end: the last one again)
      const int pair = e / S::UNITS, unit = e - pair * S::UNITS;
      wused[i] = i * 64 * kProducers + pwave * 64 < S::ITEMS; // (uniform)
      wch[i] = pair / S::OCTETS;
      wraw[i] = wch[i] * S::PITCH + pair % S::OCTETS * (8 * TAPS) + (S::BESIDE == 2 ? unit / 4 * WIN + unit % 4 * 2 : unit);
      wlast[i] = S::BESIDE == 2 && unit % 4 == 3;
      wlds[i] = unit * S::UNIT + (pair % S::OCTETS * 2 * kOC + wch[i]) * 16;
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
    auto largest = [](const auto &v, float m) {
#pragma unroll
      for (const float f : v) m = fmaxf(m, fabsf(f));
      return m;
    };
    auto produce = [&](auto splitTag) { // the operands of every step, in pieces or as they are
      constexpr bool SPLIT = decltype(splitTag)::value;
      Pieces even, odd;
      float xs = 1.0f, ws[WI], xmost[PI], wmost[WI];
      if (!SPLIT) {
        loadFilter(0, 0);
        loadFilter(atMost(1), 1);
      }
      loadPixels(even, 0);
      loadPixels(odd, atMost(1));
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * PI * CPS + RPW) : "memory"); // the filter of the first step has arrived
      __syncthreads();
      if constexpr (SPLIT) {
        constexpr int LPR = 64 / RPW; // lanes a row
        float m = 0.0f;
        const int row = pwave * RPW + lane / LPR;
#pragma unroll
        for (int i = 0; i < S::ROW; i += LPR) m = fmaxf(m, fabsf(raw[row * S::PITCH + (i + LPR <= S::ROW || i + lane % LPR < S::ROW ? i + lane % LPR : i)]));
        m = group_max<LPR>(m);
        if (lane % LPR == 0) {
          wMax[row] = __builtin_bit_cast(uint32_t, m);
          wExp[row] = scaleExponent(__builtin_bit_cast(uint32_t, m), -3);
        }
        m = 0.0f;
#pragma unroll
        for (int i = 0; i < PI; i++) {
          xmost[i] = 0.0f;
          m = largest(even.v[i], m);
        }
        m = group_max<64>(m);
        if (lane == 0) atomicMax(&xMax, __builtin_bit_cast(uint32_t, m));
        __syncthreads();
        xs = powerOf2(scaleExponent(xMax, 1));
#pragma unroll
        for (int i = 0; i < WI; i++) {
          wmost[i] = 0.0f;
          ws[i] = wused[i] ? powerOf2(wExp[wch[i]]) : 0.0f;
        }
      }
      auto put = [&](const float (&v)[8], float scale, unsigned char *at, int second) {
        if constexpr (SPLIT) {
          uint32_t hi[4], lo[4];
#pragma unroll
          for (int k = 0; k < 4; k++) splitPair(v[2 * k] * scale, v[2 * k + 1] * scale, hi[k], lo[k]);
          *reinterpret_cast<u32x4 *>(at) = u32x4{hi[0], hi[1], hi[2], hi[3]};
          *reinterpret_cast<u32x4 *>(at + second) = u32x4{lo[0], lo[1], lo[2], lo[3]};
        } else {
          constexpr int FIRST = CPS / 2; // a position's channels come half and half
          *reinterpret_cast<f32x4 *>(at) = f32x4{v[0], v[1], v[FIRST == 4 ? 2 : 4], v[FIRST == 4 ? 3 : 5]};
          *reinterpret_cast<f32x4 *>(at + second) = f32x4{v[FIRST], v[FIRST + 1], v[6], v[7]};
        }
      };
      auto putPixel = [&](const float (&v)[CPS], unsigned char *at) {
        if constexpr (CPS == 8) {
          put(v, xs, at, plane * PXB);
        } else {
          u32x2 hi, lo;
          if constexpr (SPLIT) {
            uint32_t h[2], l[2];
#pragma unroll
            for (int k = 0; k < 2; k++) splitPair(v[2 * k] * xs, v[2 * k + 1] * xs, h[k], l[k]);
            hi = u32x2{h[0], h[1]}, lo = u32x2{l[0], l[1]};
          } else {
            hi = u32x2{__builtin_bit_cast(uint32_t, v[0]), __builtin_bit_cast(uint32_t, v[1])};
            lo = u32x2{__builtin_bit_cast(uint32_t, v[2]), __builtin_bit_cast(uint32_t, v[3])};
          }
          *reinterpret_cast<u32x2 *>(at) = hi;
          *reinterpret_cast<u32x2 *>(at + plane * PXB) = lo;
        }
      };
      int slot = 0;
      auto turn = [&](Pieces &p, int s) { // what step s reads
        if (s < steps) {
          unsigned char *at = pixelBuf + (s & 1) * S::PIXELS;
#pragma unroll
          for (int i = 0; i < PI; i++) {
            if constexpr (SPLIT) xmost[i] = largest(p.v[i], xmost[i]);
            if (piece(i) < S::OCTETS * blocks) putPixel(p.v[i], at + xlds[i]);
          }
          loadPixels(p, atMost(s + 2));
          at = smem + (s & 1) * S::FILTER;
#pragma unroll
          for (int i = 0; i < WI; i++) {
            if (!wused[i]) continue;
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {
              v[k] = raw[slot * (S::RAW / 4) + wraw[i] + k % CPS * TAPS + k / CPS];
              if (k >= CPS && wlast[i]) v[k] = 0.0f;
            }
            if constexpr (SPLIT) wmost[i] = largest(v, wmost[i]);
            put(v, SPLIT ? ws[i] : 1.0f, at + wlds[i], kOC * 16);
          }
          loadFilter(atMost(s + 2), slot == 0 ? 2 : slot - 1); // (everybody is done with what was there: a step ago)
          slot = slot == 2 ? 0 : slot + 1;
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PI * CPS + RPW) : "memory"); // the filter of step s + 1 has arrived
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
      if constexpr (SPLIT) {
        // Did the pieces hold everything?  (low: there are small values; whether a window has no others is looked up only then)
        bool fault = false, low = false;
#pragma unroll
        for (int i = 0; i < PI; i++)
          if (piece(i) < S::OCTETS * blocks) {
            fault |= xmost[i] * xs >= kMost;
            low |= xmost[i] > 0.0f && xmost[i] * xs < kLeast;
          }
#pragma unroll
        for (int i = 0; i < WI; i++)
          if (wused[i]) {
            fault |= wmost[i] * ws[i] >= kMost;
            // (the scale is made for the first step's maximum, but that may be 0, or out of the scales' range)
            const float most = wMax[wch[i]] ? __builtin_bit_cast(float, wMax[wch[i]]) : wmost[i];
            fault |= most > 0.0f && most * ws[i] < kLeast;
          }
        if (fault) bad = 1;
        if (low) small = 1;
        __syncthreads();
        if (small) {
          float *maxima = reinterpret_cast<float *>(smem);
#pragma unroll
          for (int i = 0; i < PI; i++)
            if (piece(i) < S::OCTETS * blocks) maxima[piece(i) * 64 + lane] = xmost[i];
          __syncthreads();
          __syncthreads();
        }
      }
    };
    produce(std::true_type());
    if (bad) produce(std::false_type());
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
    bbase[t] = ((p.image * g.rows + p.row * g.SH - r0) * g.pitch + p.col * g.SW) * PXB + (S::OCTETS == 2 ? hl * (2 * 16) * plane : 0);
    pix[t] = q < g.pixels && col < g.OW ? p.row * g.OW + col : -1;
    img[t] = n - n0;
  }
  // The filler unit's filter values are zeros, which are taken for its pixels too (an infinity times 0 would be none).
  constexpr bool FILLED = S::UNITS % S::PAIRED != 0;
  constexpr int kFiller = S::UNITS * S::UNIT;
  if constexpr (FILLED) {
    if (tid < 2 * 64) *reinterpret_cast<u32x4 *>(smem + tid / 64 * S::FILTER + kFiller + tid % 64 * 16) = u32x4{0u, 0u, 0u, 0u};
  }
  f32x16 acc[kPT];
  auto multiply = [&](auto splitTag) -> bool { // false: the pieces did not hold everything
    constexpr bool SPLIT = decltype(splitTag)::value;
    f32x16 low[kPT]; // products with a lower piece: their roundings do not count among the others' (not SPLIT: every other product)
#pragma unroll
    for (int t = 0; t < kPT; t++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[t][i] = low[t][i] = 0.0f;
    struct Operands {
      f16x8 ah, al, bh[kPT], bl[kPT]; // not SPLIT: eight channels as two times four floats
    };
    auto read = [&](Operands &o, int step, int set) {
      const unsigned char *wat = smem + (step & 1) * S::FILTER + hl * S::HALF + l32 * 16 + set * (S::PAIRED * S::UNIT);
      const int pixelsAt = 2 * S::FILTER + (step & 1) * S::PIXELS;
      const unsigned char *xat = smem + pixelsAt;
      // (by scalars, and a selection between the lane halves)
      auto distance = [&](int unit) {
        const int ky = S::BESIDE == 2 ? unit / 4 : unit / WIN, kx = S::BESIDE == 2 ? unit % 4 * 2 : unit - ky * WIN;
        return (ky * g.DH * g.pitch + kx * g.DW) * PXB;
      };
      const int off = S::PAIRED == 2 && hl ? distance(2 * set + 1) : distance(S::PAIRED * set);
      const bool filler = FILLED && hl && set == SETS - 1;
      o.ah = *reinterpret_cast<const f16x8 *>(wat);
      o.al = *reinterpret_cast<const f16x8 *>(wat + kOC * 16);
#pragma unroll
      for (int t = 0; t < kPT; t++) {
        if constexpr (S::PAIRED == 1) {
          o.bh[t] = *reinterpret_cast<const f16x8 *>(xat + bbase[t] + off);
          o.bl[t] = *reinterpret_cast<const f16x8 *>(xat + bbase[t] + off + plane * PXB);
          continue;
        }
        const int at = filler ? kFiller : pixelsAt + bbase[t] + off, lower = at + (filler ? 0 : plane * PXB);
        if constexpr (S::BESIDE == 1) {
          o.bh[t] = *reinterpret_cast<const f16x8 *>(smem + at);
          o.bl[t] = *reinterpret_cast<const f16x8 *>(smem + lower);
        } else { // (eight bytes of either pixel; behind the last one of a row lies what is none of the window's)
          const f16x4 none = {}, *h = reinterpret_cast<const f16x4 *>(smem + at), *l = reinterpret_cast<const f16x4 *>(smem + lower);
          f16x4 h1 = h[1], l1 = l[1];
          if (hl && set % 2) h1 = none, l1 = none;
          o.bh[t] = __builtin_shufflevector(h[0], h1, 0, 1, 2, 3, 4, 5, 6, 7);
          o.bl[t] = __builtin_shufflevector(l[0], l1, 0, 1, 2, 3, 4, 5, 6, 7);
        }
      }
    };
    auto mma = [&](const Operands &o) {
      if constexpr (SPLIT) {
#pragma unroll
        for (int t = 0; t < kPT; t++) low[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(o.al, o.bh[t], low[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < kPT; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(o.ah, o.bh[t], acc[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < kPT; t++) low[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(o.ah, o.bl[t], low[t], 0, 0, 0);
      } else {
        // (a step of two products has one of either lane half: channel k and channel 8 + k)
#pragma unroll
        for (int k = 0; k < 8; k++) {
          const float a = __builtin_bit_cast(f32x4, k < 4 ? o.ah : o.al)[k % 4];
#pragma unroll
          for (int t = 0; t < kPT; t++)
            (k % 2 ? low : acc)[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, __builtin_bit_cast(f32x4, k < 4 ? o.bh[t] : o.bl[t])[k % 4], (k % 2 ? low : acc)[t], 0, 0, 0);
        }
      }
    };
    __syncthreads();
    if constexpr (SPLIT) __syncthreads();
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
        mma(even);
        read(even, s, set + 2 * KS < SETS ? set + 2 * KS : from);
        mma(odd);
      }
      if (set < SETS) mma(even);
      __syncthreads();
    }
    if constexpr (SPLIT) {
      __syncthreads();
      const int xe = scaleExponent(xMax, 1);
      if (small) {
        __syncthreads();
        const float *maxima = reinterpret_cast<const float *>(smem);
        bool fault = false;
#pragma unroll
        for (int t = 0; t < kPT; t++) {
          float m = 0.0f;
          const int base = bbase[t] / PXB - (S::OCTETS == 2 ? hl * plane : 0); // (a lane half has a plane of pixels and one of lower pieces each)
          for (int ky = 0; ky < WIN; ky++)
            for (int kx = 0; kx < WIN; kx++) m = fmaxf(m, maxima[base + ky * g.DH * g.pitch + kx * g.DW]);
          m = halves_max(m);
          fault |= pix[t] >= 0 && m > 0.0f && m * powerOf2(xe) < kLeast;
        }
        if (fault) bad = 1;
        __syncthreads();
      }
      if (bad) return false;
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int down = -xe - wExp[8 * (i / 4) + 4 * hl + i % 4];
#pragma unroll
        for (int t = 0; t < kPT; t++) acc[t][i] = ldexpf(acc[t][i] + low[t][i], down);
      }
    } else {
#pragma unroll
      for (int t = 0; t < kPT; t++) acc[t] += low[t];
    }
    return true;
  };
  if (!multiply(std::true_type())) multiply(std::false_type());

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

// The tiles, and what a launch in them takes: us = start + rounds of the CUs * (block + step * steps), fitted to 800 launches of
// each of the larger two of 3 x 3, 450 and 280 of the others (a tenth to a ninetieth percentile of 0.93 to 1.08 times what was measured), and
// to some 40 each of 5 x 5 and 7 x 7 (0.95 to 1.04).
struct SplitTile {
  int pixels, cap;
  double start, block, step;
};
constexpr SplitTile kTiles[] = {{64, 256, 1.5, 4.7, 0.89}, {64, 512, 1.5, 5.1, 1.08}, {128, 256, 1.4, 5.5, 1.10}, {128, 512, 1.3, 6.0, 1.20}, {256, 512, 0.7, 7.5, 1.42},
                                {64, 384, 1.2, 4.6, 1.085}, {128, 384, 1.2, 5.1, 1.49}, {64, 704, 1.1, 4.85, 1.247}, {128, 704, 0.75, 5.7, 1.55}};
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
  case 1: launch(conv_split_kernel<3, 4, 512>); break;
  case 2: launch(conv_split_kernel<3, 2, 256>); break;
  case 3: launch(conv_split_kernel<3, 2, 512>); break;
  case 4: launch(conv_split_kernel<3, 1, 512>); break;
  case 5: launch(conv_split_kernel<5, 4, 384>); break;
  case 6: launch(conv_split_kernel<5, 2, 384>); break;
  case 7: launch(conv_split_kernel<7, 4, 704>); break;
  default: launch(conv_split_kernel<7, 2, 704>);
  }
  return true;
}

} // namespace mgpu
