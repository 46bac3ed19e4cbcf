// C++ entry points behind the extern "C" layer (c_api.cpp) and the template
// wrappers of Kernels/GPU/Ops.h.  All of them enqueue on `stream` and throw
// std::logic_error (after printing) on bad arguments or a failed launch.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace mgpu {

enum class DType { F32 = 0, F16 = 1, BF16 = 2 };

void addF32(const float *a, const float *b, float *c, int64_t n, hipStream_t stream);

// residual may be null (plain LayerNorm); sumOut may be null (the rounded sum is then not written).
void layerNorm(DType dt, const void *input, const void *residual, const void *gamma,
               const void *beta, void *sumOut, void *normed, float eps, int m, int n,
               hipStream_t stream);

// castOut = fp16(input), normed = LayerNorm(castOut) in one pass over fp32 rows
// (n a multiple of 8 up to 4096, 16-byte aligned operands); false, with
// nothing enqueued, for other shapes.
bool castLayerNormF32ToF16(const float *input, const void *gamma, const void *beta, void *castOut, void *normed,
                           float eps, int m, int n, hipStream_t stream);

void fusedMHA(DType dt, const void *qkv, const int32_t *seqlens, void *out, int B, int S, int H,
              int D, float scale, bool causal, hipStream_t stream);

// The reference's form of the sequence lengths: B + 1 prefix sums over token
// rows packed back to back (qkv [total, 3, H, D], out [total, H * D]); maxS
// bounds the longest sequence.
void fusedMHACuSeqlens(DType dt, const void *qkv, const int32_t *cuSeqlens, void *out, int B, int maxS, int H,
                       int D, float scale, bool causal, hipStream_t stream);
// The kernel whose wavefronts split the keys (fmha_split.hip), on operands that fusedMHA has checked; false, and nothing
// launched, where its rule leaves the call to the 128-query kernel.
bool fusedMHASplitKeys(DType dt, const void *qkv, const int32_t *seqlens, const int32_t *cuSeqlens, void *out, int B, int S,
                       int H, int D, float scale, bool causal, hipStream_t stream);

void castF32ToF16(void *dst, const float *src, size_t size, hipStream_t stream);
void castF16ToF32(float *dst, const void *src, size_t size, hipStream_t stream);
void castF32ToBF16(void *dst, const float *src, size_t size, hipStream_t stream);
void castBF16ToF32(float *dst, const void *src, size_t size, hipStream_t stream);
// dst[c][r] = src[r][c] of a row-major rows x cols matrix (fp32 -> fp16; any 16-bit type, bit for bit)
void transposeCastF32ToF16(void *dst, const float *src, int64_t rows, int64_t cols, hipStream_t stream);
void transpose16(void *dst, const void *src, int64_t rows, int64_t cols, hipStream_t stream);
// LayerNorm of the sum of fp16 rows, rounded to fp16, in fp32 (m, n > 0); false, and nothing launched, for rows that are not whole aligned vectors or too wide.
bool layerNormF16ToF32(const void *input, const void *residual, const void *gamma, const void *beta, float *normed, float eps, int m, int n,
                       hipStream_t stream);
// fp32 arrays to fp16, up to kMaxCastJobs of them in one launch; kMajor: dst[c][r] = src[r][c].
struct CastJob {
  const float *src;
  void *dst;
  int64_t rows, cols;
  bool kMajor;
  bool vector; // (set by the call: 16-byte accesses allowed)
};
constexpr int kMaxCastJobs = 8;
void castWeightsF32ToF16(CastJob *jobs, int count, hipStream_t stream);
// The same and castLayerNormF32ToF16 (m, n > 0) in one launch; false, and nothing launched, where that one would be.
bool castWeightsLayerNormF32ToF16(CastJob *jobs, int count, const float *input, const void *gamma, const void *beta, void *castOut,
                                  void *normed, float eps, int m, int n, hipStream_t stream);
void fillF16(void *dst, size_t count, float value, hipStream_t stream);
void fillI32(int32_t *dst, size_t count, int32_t value, hipStream_t stream);

void addFusedQKVBiasTranspose(DType dt, void *q, void *k, void *v, void *qkv, const void *bias, int B, int S,
                              int tokens, int H, int D, hipStream_t stream);
void addFusedQKVBiasTransposeF16(void *q, void *k, void *v, void *qkv, const void *bias, int B,
                                 int S, int tokens, int H, int D, hipStream_t stream);

enum Activation { ACT_NONE = 0, ACT_RELU = 1, ACT_GELU = 2 };
void gemmInit();
void gemmDeinit();
// weightKMajor: the weight is stored [N, K] (each output column's K values contiguous) instead of
// the ABI's [K, N]; the layers' weight cache keeps such copies, which the library multiplies
// faster.  Served by the library or, few tiles, by gemm_ksplit.
void matmulEx(DType dt, const void *input, const void *weight, const void *bias, void *output,
              const void *residual, int64_t M, int64_t N, int64_t K, bool hasBias, int act,
              bool hasResidual, hipStream_t stream, bool weightKMajor = false);
// fp16 operands, in . weight + bias + residual in fp32 on the kernel that matmulEx would run (rounded to fp16 on the way, except by
// gemm_wide); false, and nothing launched, where that one has no such epilogue.
bool matmulResidualF32(const void *input, const void *weight, const void *bias, const void *residual, float *output, int64_t M, int64_t N,
                       int64_t K, bool weightKMajor, hipStream_t stream);
// Which kernel matmulEx runs a product on (K, N > 0; 16-byte aligned operands), and the width at which gemm_wide serves it, 0 where
// it does not.
enum class GemmKernel { Library, Mfma, KSplit, F32Small, Wide, Round };
GemmKernel gemmKernelFor(DType dt, int64_t M, int64_t N, int64_t K, bool hasBias, int act, bool hasResidual, bool weightKMajor);
int gemmWideWidth(DType dt, int64_t M, int64_t N, int64_t K, int act, bool hasResidual);
// Should a caller that can keep a K-major copy of the weight hand that one to matmulEx for this
// problem?  (The committed table, else: wherever the library would serve it as it is.)
bool gemmPrefersKMajor(DType dt, const void *weight, const void *bias, int64_t M, int64_t N, int64_t K, bool hasBias, int act,
                       bool hasResidual);
// Would a caller that makes its fp16 weight anew on every call, in either layout at the same price, rather
// have it K-major?
bool gemmWantsKMajorCast(DType dt, int64_t M, int64_t N, int64_t K, bool hasBias, int act, bool hasResidual);

// Hand-written MFMA GEMM (gemm_mfma.hip): fp16 / bf16, M a multiple of 128, N of
// 128 or 96, K of 32, 16-byte aligned operands; bias and residual may be null.
bool gemmMfmaSupports(DType dt, const void *in, const void *weight, const void *bias, const void *residual,
                      const void *out, int64_t M, int64_t N, int64_t K);
void gemmMfma(DType dt, const void *in, const void *weight, const void *bias, const void *residual, void *out,
              int64_t M, int64_t N, int64_t K, int act, hipStream_t stream);

// The same kernel where its tiles overhang the shape: any M, N a multiple of 8, K of 32.
bool gemmMfmaSupportsRagged(DType dt, const void *in, const void *weight, const void *bias, const void *residual,
                            const void *out, int64_t M, int64_t N, int64_t K);
// gemmMfmaKernel: which of gemm_round, gemm_wide and the kernel itself runs it there, and the width of the tiles; gemmMfmaShallow:
// is the product so shallow that the kernel itself is ahead of the other two; gemmMfmaCost: the estimated us on a shape, on the
// scale of gemmKSplitBest.
bool gemmMfmaShallow(int64_t M, int64_t N, int64_t K, int act, bool hasResidual);
GemmKernel gemmMfmaKernel(DType dt, const void *in, const void *weight, const void *bias, const void *residual, const void *out, int64_t M,
                          int64_t N, int64_t K, int act, int *width);
double gemmMfmaCost(int64_t M, int64_t N, int64_t K, int act, bool hasResidual = false);
void gemmMfmaRagged(DType dt, const void *in, const void *weight, const void *bias, const void *residual, void *out,
                    int64_t M, int64_t N, int64_t K, int act, hipStream_t stream);

// Tiles of 256 rows, one block per CU (gemm_wide.hip): fp16 / bf16, any M, N and K multiples of 8, K from 72 on.
// width: 128, 192 or 256 columns; gemmWideBest: the width for a shape and its estimated us, on the scale of gemmKSplitBest.
int gemmWideBest(int64_t M, int64_t N, int64_t K, int act, bool hasResidual, double *cost);
bool gemmWideSupports(DType dt, const void *in, const void *weight, const void *bias, const void *residual, const void *out, int64_t M,
                      int64_t N, int64_t K);
void gemmWide(DType dt, const void *in, const void *weight, const void *bias, const void *residual, void *out, int64_t M, int64_t N,
              int64_t K, int act, int width, hipStream_t stream);
// fp16 operands, in . weight + bias + residual in fp32.
void gemmWideResidualF32(const void *in, const void *weight, const void *bias, const void *residual, float *out, int64_t M, int64_t N, int64_t K,
                         int width, hipStream_t stream);

// At most one tile of 128 x 96 or 128 x 128 per CU (gemm_round.hip): N and K multiples of 8; planes: K of 64.  gemmRoundWidth: the width
// for a shape, 0 where it does not go.
int gemmRoundWidth(DType dt, const void *in, const void *weight, const void *bias, const void *residual, const void *out, int64_t M, int64_t N,
                   int64_t K);
void gemmRound(DType dt, const void *in, const void *weight, const void *bias, const void *residual, void *out, int64_t M, int64_t N,
               int64_t K, int act, int width, hipStream_t stream);
void gemmRoundResidualF32(const void *in, const void *weight, const void *bias, const void *residual, float *out, int64_t M, int64_t N, int64_t K,
                          int width, hipStream_t stream);
void gemmRoundPartialF16(const void *in, const void *weight, float *planes, int64_t M, int64_t N, int64_t K, int width, int parts,
                         hipStream_t stream);

// Small tiles, the reduction split over a block's wavefronts (gemm_ksplit.hip): fp16 / bf16, any M, N and K
// multiples of 8.  gemmKSplitBest: the tile for a shape and its estimated us, to compare with the others.
enum class KSplitTile { T32x32, T32x64, T64x64 };
KSplitTile gemmKSplitBest(int64_t M, int64_t N, int64_t K, int act, double *cost, int parts = 1);
bool gemmKSplitSupports(DType dt, const void *in, const void *weight, const void *bias, const void *residual, const void *out, int64_t M,
                        int64_t N, int64_t K);
void gemmKSplit(DType dt, const void *in, const void *weight, const void *bias, const void *residual, void *out, int64_t M, int64_t N,
                int64_t K, int act, KSplitTile tile, bool weightKMajor, hipStream_t stream);
void gemmKSplitResidualF32(const void *in, const void *weight, const void *bias, const void *residual, float *out, int64_t M, int64_t N,
                           int64_t K, KSplitTile tile, bool weightKMajor, hipStream_t stream);
// A GEMM whose reduction is split over blocks: `parts` fp32 planes [M, N] of partial sums (16-byte aligned), added up by
// one of the kernels of partial_sums.hip.  gemmPartialPlan: parts = 0 where the shape is better served whole.
struct PartialPlan {
  int parts = 0;
  bool mfma = false; // gemm_mfma, else gemm_ksplit on `tile`
  KSplitTile tile = KSplitTile::T32x32;
};
PartialPlan gemmPartialPlan(const void *in, const void *weight, int64_t M, int64_t N, int64_t K, bool weightKMajor);
void gemmPartialF16(const PartialPlan &plan, const void *in, const void *weight, float *planes, int64_t M, int64_t N, int64_t K, hipStream_t stream);
double gemmMfmaPartialCost(int64_t M, int64_t N, int64_t K, int parts);
void gemmMfmaPartialF16(const void *in, const void *weight, float *planes, int64_t M, int64_t N, int64_t K, int parts, hipStream_t stream);
void gemmKSplitPartialF16(const void *in, const void *weight, float *planes, int64_t M, int64_t N, int64_t K, KSplitTile tile, int parts,
                          hipStream_t stream);
// The sum of the planes + bias + residual: through a LayerNorm (fp16; the rounded sum to sumOut when not null; or fp32), or as it
// is, in fp32.  partialSumsSupports: widths and alignment.
bool partialSumsSupports(const void *bias, const void *residual, const void *gamma, const void *beta, const void *out, int64_t M, int64_t N);
void partialSumsLayerNormF16(const float *planes, int parts, const void *bias, const void *residual, const void *gamma, const void *beta,
                             void *sumOut, void *out, float eps, int64_t M, int64_t N, hipStream_t stream);
void partialSumsLayerNormF32(const float *planes, int parts, const void *bias, const void *residual, const void *gamma, const void *beta,
                             float *out, float eps, int64_t M, int64_t N, hipStream_t stream);
void partialSumsF32(const float *planes, int parts, const void *bias, const void *residual, float *out, int64_t M, int64_t N,
                    hipStream_t stream);
// fp32, any shape, for few tiles (gemm_f32_small.hip).
void gemmF32Small(const float *in, const float *weight, const float *bias, const float *residual, float *out, int64_t M, int64_t N, int64_t K,
                  int act, hipStream_t stream);

void conv2d(const float *input, const float *weight, const float *bias, float *output, const float *postAdd,
            int64_t N, int64_t IC, int64_t H, int64_t W, int64_t OC, int64_t KH, int64_t KW, int64_t OH,
            int64_t OW, int64_t PHL, int64_t PWL, int64_t PHR, int64_t PWR, int64_t SH, int64_t SW, int64_t DH,
            int64_t DW, bool hasPostAdd, bool relu, hipStream_t stream);
// How many wavefronts share a tile of its kernel that stages the filter in LDS, 0 where another one serves the convolution (win: the
// window's side; pixels: of the output, of all images).
int convStagedWaves(int win, int64_t stride, int64_t pixels, int64_t IC, int64_t OC, int64_t OW, int64_t cus);
// Do patches of input rows in LDS serve a square convolution (rowTiles: tiles of 32 pixels of one output row by 32 channels)?
bool convByPatches(int win, int stride, int64_t tiles, int64_t rowTiles, int64_t IC, int64_t OC, int64_t OW, int64_t cus);
// How long the kernels above take for a 3 x 3 convolution, in us (see conv.hip).
double convWindowTime(int64_t stride, int64_t pixels, int64_t IC, int64_t OC, int64_t OW, int64_t cus);
// 3 x 3, 5 x 5 and 7 x 7 on the bf16 matrix cores in three bf16 numbers (conv_split.hip), of channels that are a multiple of 16, 8 and 4: the
// tile and the strips of columns that take the least time (strips 0: none less than `limit` us), and the launch (false: not for these
// sizes or pointers).
struct ConvSplitPlan {
  int tile, strips;
  double us;
};
ConvSplitPlan convSplitPlan(int N, int IC, int OC, int OH, int OW, int SH, int SW, int DH, int DW, int cus, double limit);
ConvSplitPlan convSplitPlan5(int N, int IC, int OC, int OH, int OW, int SH, int SW, int DH, int DW, int cus, double limit);
ConvSplitPlan convSplitPlan7(int N, int IC, int OC, int OH, int OW, int SH, int SW, int DH, int DW, int cus, double limit);
bool convSplit(const ConvSplitPlan &plan, const float *x, const float *w, const float *bias, float *y, const float *add, int64_t N, int64_t IC,
               int64_t H, int64_t W, int64_t OC, int64_t OH, int64_t OW, int64_t PHL, int64_t PWL, int64_t SH, int64_t SW, int64_t DH,
               int64_t DW, bool relu, hipStream_t stream);
// How long the same take for 3 x 3, 5 x 5 or 7 x 7 on few tiles, in us; 0: not few.
double convFewTilesTime(int win, int64_t stride, int64_t pixels, int64_t IC, int64_t OC, int64_t OW, int64_t cus);
// 3 x 3, 5 x 5 or 7 x 7 on tiles of 16 pixels (conv_small.hip), from channels that are a multiple of 4: the output channels of a tile, 16 or 32, that
// take the least time (0: none) and the launch (false: not for these sizes).
struct ConvSmallPlan {
  int ocSide;
  double us;
};
ConvSmallPlan convSmallPlan(int win, int64_t pixels, int64_t IC, int64_t OC, int64_t cus);
bool convSmall(int win, int ocSide, const float *x, const float *w, const float *bias, float *y, const float *add, int64_t N, int64_t IC, int64_t H, int64_t W,
               int64_t OC, int64_t OH, int64_t OW, int64_t PHL, int64_t PWL, int64_t SH, int64_t SW, int64_t DH, int64_t DW, bool relu,
               hipStream_t stream);
void pool2d(const float *input, float *output, int64_t N, int64_t C, int64_t H, int64_t W, int64_t OH, int64_t OW,
            int64_t KH, int64_t KW, int64_t PHL, int64_t PWL, int64_t PHR, int64_t PWR, int64_t SH, int64_t SW,
            int64_t method, hipStream_t stream);

void llmInit();
void llmDeinit();
// Opt-in fp16 cache of the reference layer's fp32 weights (see llm.cpp); false also drops the copies.
void llmCacheWeights(bool enable);
void decodingContextLayer(float *input, float *qkv, float *gemm_weight, float *gemm_bias,
                          float *ffn1_weight, float *ffn1_bias, float *ffn2_weight,
                          float *ffn2_bias, float *output, int64_t batch, int64_t seq_len,
                          int64_t d_model, int64_t ffn, int64_t heads, bool norm_first,
                          bool causal, bool relu, hipStream_t stream);

void bertEncoderLayerF16(const void *x, const void *wqkv, const void *bqkv, const void *wo,
                         const void *bo, const void *gamma1, const void *beta1, const void *w1,
                         const void *b1, const void *w2, const void *b2, const void *gamma2,
                         const void *beta2, const int32_t *seqlens, void *out, int64_t B,
                         int64_t S, int64_t d, int64_t ffn, int64_t H, float eps,
                         hipStream_t stream);

// The same layer with every temporary in a fixed file-scope device array
// (layer_noalloc.hip): no allocation, no library GEMM; shapes beyond the array
// or outside the hand-written GEMM's tiling are an error.
void noAllocInit();
size_t noAllocScratchBytes();
void bertEncoderLayerF16NoAlloc(const void *x, const void *wqkv, const void *bqkv, const void *wo,
                                const void *bo, const void *gamma1, const void *beta1, const void *w1,
                                const void *b1, const void *w2, const void *b2, const void *gamma2,
                                const void *beta2, const int32_t *seqlens, void *out, int64_t B,
                                int64_t S, int64_t d, int64_t ffn, int64_t H, float eps,
                                hipStream_t stream);

void geluInPlaceF16(void *data, size_t n, hipStream_t stream);
void geluInPlaceBF16(void *data, size_t n, hipStream_t stream);
void geluInPlaceF32(float *data, size_t n, hipStream_t stream);

} // namespace mgpu
