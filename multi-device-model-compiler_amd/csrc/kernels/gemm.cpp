// GEMM with bias / activation / residual epilogue over hipBLASLt.
//
// Replaces mgpuMatmul and mgpuMatmulEx<T> (lib/Kernels/GPU/Ops.cu:57-120,
// 134-234).  Same row-major contract through the column-major operand swap of
// Ops.cu:83-85,178-183: out^T[N,M] = W^T[N,K] . in^T[K,M].  Differences:
//  * the whole plan (operation descriptor, layouts, chosen algorithm) is built
//    once per (shape, flags, type) and reused; the reference rebuilds all
//    descriptors on every call and caches only the heuristic result;
//  * fp16 / bf16 inputs accumulate in fp32 (HIPBLAS_COMPUTE_32F); the reference
//    asks for fp16 accumulation (Ops.cu:164-167);
//  * GELU is applied by an exact-erf kernel after a bias-only epilogue, because
//    the library's fused GELU is the tanh approximation;
//  * a call only enqueues: which of the kernels serves a shape - the library or
//    a hand-written one (gemm_wide.hip, gemm_round.hip, gemm_mfma.hip, gemm_ksplit.hip, gemm_f32_small.hip) -
//    is a fixed rule: gemm_wide and gemm_round first, where they apply; for the rest a
//    table decided offline (gemm_table.inc, written by `bench.py --tune-gemm`
//    from measurements on an MI355X) and, for shapes the table does not hold,
//    lines on the shape; the library runs the heuristic's first algorithm.
//    MGPU_GEMM_KERNEL=library or =mfma in the environment overrides both.
//    Nothing in this library measures anything: the tuner that writes the
//    table lives with the benchmark's launch loops;
//  * the library's workspace is per caller stream (allocated on a stream's
//    first library GEMM outside a capture), so GEMMs on different streams never
//    share one; a stream first seen under capture gets an algorithm that needs
//    no workspace.
#include "common.hpp"
#include "mgpu_ops_internal.hpp"

#include <hipblaslt/hipblaslt.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

namespace mgpu {

namespace {

hipblasLtHandle_t ltHandle = nullptr;
constexpr size_t workspaceSize = 32u * 1024u * 1024u;
std::mutex planMutex;
std::map<hipStream_t, void *> workspaceOf; // per caller stream, see the header comment

bool isCapturing(hipStream_t s) {
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(s, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone;
}

// The stream's workspace; null when it has none yet and none can be made now (the stream
// is capturing, or the allocation failed).  Workspaces are kept per stream handle until
// gemmDeinit(); a caller that creates and destroys streams without end should run its
// GEMMs on a bounded set of them.
void *workspaceFor(hipStream_t s) {
  auto it = workspaceOf.find(s);
  if (it != workspaceOf.end()) return it->second;
  if (isCapturing(s)) return nullptr;
  void *ws = nullptr;
  if (hipMalloc(&ws, workspaceSize) != hipSuccess) { // out of memory, or another stream is capturing
    (void)hipGetLastError();
    return nullptr; // the caller falls back to an algorithm that needs no workspace; asked again next time
  }
  workspaceOf[s] = ws;
  return ws;
}

void checkBlas(hipblasStatus_t status, const char *where) {
  if (status != HIPBLAS_STATUS_SUCCESS)
    fail(std::string(where) + ": hipBLASLt API failed with status " + std::to_string((int)status));
}
#define MGPU_CHECK_BLAS(expr) checkBlas((expr), #expr)

struct Plan {
  hipblasLtMatmulDesc_t op = nullptr;
  hipblasLtMatrixLayout_t a = nullptr, b = nullptr, d = nullptr;
  hipblasLtMatmulAlgo_t algo;          // the heuristic's first answer (or the tuned one)
  size_t algoWorkspace = 0;
  hipblasLtMatmulAlgo_t algoNoWs;      // the first answer that needs no workspace
  bool hasNoWs = false;
};

// Shapes decided offline: {type (1 fp16, 2 bf16), M, N, K, hasBias, act, hasResidual, hand-written kernel
// (against the library, both on the ABI's [K, N] weight)?, the library on a K-major copy of the weight
// ahead of both?}.
struct TableEntry {
  int dt;
  int64_t M, N, K;
  int hasBias, act, hasResidual, handWritten, kMajorLibrary;
};
const TableEntry kTable[] = {
#include "gemm_table.inc"
    {0, 0, 0, 0, 0, 0, 0, 0, 0}}; // (no product has no rows)

// 128 x 128 tiles of a shape: up to one per CU every form of the hand-written kernels pays.
int64_t tiles128(int64_t M, int64_t N) { return (M + 127) / 128 * ((N + 127) / 128); }

// Where the library, on a [K, N] weight, is ahead of gemm_ksplit and of what gemm_mfma's launcher has, for products that gemm_wide and
// gemm_round (wideWidth, raggedRoundWidth) do not take (us, library / gemm_mfma or, small, gemm_ksplit):
//  * up to one round of the CUs nowhere (2000 x 2000 x 1024 17.7 / 13.7), but for fewer than 128 rows: those tiles read the weight no
//    faster for it: 32 x 20000 x 512 8.8 / 7.9, x 1024 10.8 / 12.2, 8 x 16384 x 2048 13.2 / 14.6, 1 x 33024 x 1024 13.8 / 16.8, but 8 x
//    16384 x 1024 8.6 / 5.7, 1 x 12288 x 4096 21.3 / 20.2; with a GELU, a pass of its own behind the library, later;
//  * beyond, 64 deep at most: from 400 tiles that overhang on; and what is too large for gemm_wide, which is deep or wide.
bool libraryAhead(int64_t M, int64_t N, int64_t K, int act, bool aligned) {
  const int64_t tiles = tiles128(M, N);
  if (M < 128 && act != ACT_GELU) return tiles > 128 && tiles > 100000 / K;
  if (tiles <= numComputeUnits()) return false;
  if (act == ACT_GELU) return tiles > 1400000 / K;
  return K > 1024 || (tiles > 400 && !aligned);
}

// 0: measure, 1: always the library, 2: the hand-written kernel wherever it applies
int forcedKernel() {
  static const int mode = [] {
    const char *v = std::getenv("MGPU_GEMM_KERNEL");
    if (!v) return 0;
    if (!std::strcmp(v, "library")) return 1;
    if (!std::strcmp(v, "mfma")) return 2;
    return 0;
  }();
  return mode;
}

bool mfmaShape(DType dt, int64_t M, int64_t N, int64_t K) {
  return (dt == DType::F16 || dt == DType::BF16) && M > 0 && M % 128 == 0 && (N % 128 == 0 || N % 96 == 0) && K % 32 == 0;
}

const TableEntry *tableRow(DType dt, int64_t M, int64_t N, int64_t K, bool hasBias, int act, bool hasResidual) {
  for (const TableEntry &e : kTable)
    if (e.dt == (int)dt && e.M == M && e.N == N && e.K == K && e.hasBias == (int)hasBias && e.act == act &&
        e.hasResidual == (int)hasResidual)
      return &e;
  return nullptr;
}

// The width at which gemm_wide serves a call, 0 where it does not.  Beyond one round of 128 x 128 tiles it is ahead of
// everything else - over 550 such shapes the library takes 1.19 to 1.38 times as long (by the number of tiles; never less
// than 0.96), gemm_mfma's paired schedule before it 1.19 to 1.31 (us, library / gemm_mfma / gemm_wide: 4096 x 3072 x 768 + GELU
// 37 / 28.2 / 24.6, 4096 x 6144 x 2048 107 / 109 / 88.5, 3000 x 2304 x 2048 36.6 / 36.6 / 27.4).  Up to one round gemm_round's
// smaller tiles are (609 shapes: gemm_wide the best of all in 14, by 8 % at most) - but not where they would take more than four
// fifths of the CUs on a product of middling depth, which some cards slow down (see gemmWideBest; us there, gemm_mfma before / gemm_round /
// half as many tiles of 256 x 128: 2048 x 2048 x 512 10.7 / 12.0 / 8.2, x 1024 14.8 / 15.8 / 12.5, 4096 x 1024 x 512 9.7 / 11.7 / 8.0; x 256 6.8 / 5.9
// and 2048 x 2048 x 2048 23.1 / 23.8 stay).  Fewer than 128 rows would leave more than half of every tile empty.
int wideWidth(DType dt, const void *in, const void *weight, const void *bias, const void *residual, const void *out, int64_t M, int64_t N,
              int64_t K, int act) {
  const int64_t cus = numComputeUnits(), tiles = tiles128(M, N);
  const bool crowded = tiles <= cus && tiles * 5 > cus * 4 && K >= 384 && K <= 1408 && act != ACT_GELU;
  if ((tiles <= cus && !crowded) || M < 128 || forcedKernel() || !gemmWideSupports(dt, in, weight, bias, residual, out, M, N, K)) return 0;
  double cost;
  const int width = gemmWideBest(M, N, K, act, residual != nullptr, &cost);
  return !crowded || cost < gemmMfmaCost(M, N, K, act) + 3.0 ? width : 0;
}

// What gemmMfmaCost answers at least, for gemm_round and for any of its kernels: a call of few tiles is decided without it (155 -> 65 ns of
// the 2.8 us that a call takes the host).
constexpr double kRoundLeast = 3.2, kMfmaLeast = 2.4;

// And gemm_round's where the depth is no multiple of 64, which it fills up with zeros (us, what ran before - the library, or gemm_mfma at
// multiples of 32 - / gemm_round: 512 x 3072 x 72 10.5 / 4.6, x 296 10.4 / 5.6, x 1000 16.1 / 10.5, x 3000 30.9 / 23.6; 3000 x 1000 x 520 15.6 /
// 10.3; x 96 6.0 / 6.4, x 1376 18.3 / 17.0).  Where gemm_ksplit's estimate is lower it stays: 500 x 2000 x 1000 9.6 / 9.6.  gemm_wide, the
// same: 4261 x 1064 x 1000 28.4 / 18.4, 6000 x 3000 x 520 49.9 / 31, 4096 x 3080 x 296 33.0 / 16.9, x 160 26.1 / 13.6.
int raggedRoundWidth(DType dt, const void *in, const void *weight, const void *bias, const void *residual, const void *out, int64_t M, int64_t N,
                     int64_t K, int act, double kSplitCost) {
  if (K % 64 == 0 || dt == DType::F32 || kSplitCost <= kRoundLeast || forcedKernel()) return 0;
  const int width = gemmRoundWidth(dt, in, weight, bias, residual, out, M, N, K);
  if (!width || gemmMfmaShallow(M, N, K, act, residual)) return 0;
  return gemmMfmaCost(M, N, (K + 63) / 64 * 64, act) < kSplitCost ? width : 0;
}

// The kernel for a call, decided without a lookup of the library's plans (a library call costs 6-7 us of
// host time, a hand-written one a launch).
//  * fp32: the small kernel by tiles of 32 x 32 times k, as its calls cross those of the library (us a call, library /
//    small: 256 x 512 10.9 / 6.0, 768 x 256 10.9 / 8.6, 3072 x 64 12.3 / 11.0, 2160 x 129 17.3 / 13.3, 768 x 400 10.6 / 11.9, 3072 x
//    129 16.9 / 17.5, 12288 x 32 20.3 / 28.2; 7 x 768 23.9 / 6.6, 256 x 768 14.5 / 7.8, 128 x 1024 10.1 / 8.7, 7 x 1536 10.0 / 11.0).  With a GELU, which is a pass of its own behind the library, further the shorter
//    the reduction: 23500 x 64 95 / 76, 12288 x 129 64 / 60, 3072 x 256 31.4 / 27.5, 2160 x 400 33.8 / 30.8, 768 x 512 14.2 / 13.7, but
//    23500 x 129 115 / 119, 3072 x 400 38.6 / 39.7, 2160 x 512 34.7 / 37.2.
//  * fp16 / bf16: the aligned shapes of the table as it says; otherwise the library where libraryAhead says so, else the
//    cheaper of gemm_mfma and gemm_ksplit by their estimates.
//  * K-major weights: gemm_ksplit while its tiles are at most one round of the CUs, two of a reduction up to 512
//    deep (us a call, library / gemm_ksplit, tiles of 64 x 64 times k: 414 x 80 10.7 / 6.9, 512 x 256 11.1 / 8.0, 512 x 384
//    10.6 / 9.9, 414 x 512 11.1 / 10.6, but 414 x 768 10.5 / 12.8 and 1424 x 64 11.2 / 17.9); beyond, the library, for
//    which the layout was made.
struct Choice {
  GemmKernel kernel;
  int width = 0; // of a tile of gemm_wide or gemm_round
  KSplitTile tile = KSplitTile::T32x32; // of gemm_ksplit
};
Choice chooseKernel(DType dt, const void *in, const void *weight, const void *bias, const void *residual, const void *out, int64_t M,
                    int64_t N, int64_t K, bool hasBias, int act, bool hasResidual, bool weightKMajor) {
  if (forcedKernel() == 1) return {GemmKernel::Library};
  if (dt == DType::F32) {
    const int64_t tiles = (M + 31) / 32 * ((N + 31) / 32);
    const int64_t most = act != ACT_GELU || K > 512 ? 200000 : K <= 128 ? 1500000 : K <= 400 ? 800000 : 300000;
    return !forcedKernel() && !weightKMajor && K <= 1024 && tiles <= most / K ? Choice{GemmKernel::F32Small} : Choice{GemmKernel::Library};
  }
  const bool kSplitOk = gemmKSplitSupports(dt, in, weight, bias, residual, out, M, N, K);
  double kSplitCost = 0.0;
  const KSplitTile tile = gemmKSplitBest(M, N, K, act, &kSplitCost);
  if (weightKMajor) {
    const int64_t bm = tile == KSplitTile::T64x64 ? 64 : 32, bn = tile == KSplitTile::T32x32 ? 32 : 64;
    const int64_t most = (K <= 512 ? 2 : 1) * (int64_t)numComputeUnits();
    return kSplitOk && !forcedKernel() && (M + bm - 1) / bm * ((N + bn - 1) / bn) <= most ? Choice{GemmKernel::KSplit, 0, tile} : Choice{GemmKernel::Library};
  }
  const bool mfmaOk = gemmMfmaSupportsRagged(dt, in, weight, bias, residual, out, M, N, K);
  auto mfma = [&] {
    Choice c;
    c.kernel = gemmMfmaKernel(dt, in, weight, bias, residual, out, M, N, K, act, &c.width);
    return c;
  };
  if (const int width = wideWidth(dt, in, weight, bias, residual, out, M, N, K, act))
    return mfmaOk && gemmMfmaShallow(M, N, K, act, residual) ? mfma() : Choice{GemmKernel::Wide, width};
  if (const int width = raggedRoundWidth(dt, in, weight, bias, residual, out, M, N, K, act, kSplitCost)) return {GemmKernel::Round, width};
  if (forcedKernel() == 2) return mfmaShape(dt, M, N, K) && mfmaOk ? mfma() : Choice{GemmKernel::Library};
  const bool aligned = mfmaOk && mfmaShape(dt, M, N, K);
  if (aligned)
    if (const TableEntry *e = tableRow(dt, M, N, K, hasBias, act, hasResidual)) return e->handWritten ? mfma() : Choice{GemmKernel::Library};
  if (libraryAhead(M, N, K, act, aligned)) return {GemmKernel::Library};
  if (kSplitOk && kSplitCost <= kMfmaLeast) return {GemmKernel::KSplit, 0, tile};
  const double mfmaCost = gemmMfmaCost(M, N, K, act, hasResidual);
  if (mfmaOk && mfmaCost < kSplitCost) return mfma();
  // (where gemm_mfma cannot go - K no multiple of 32 - its estimate stands for the library's time)
  return kSplitOk && kSplitCost < 1.2 * mfmaCost ? Choice{GemmKernel::KSplit, 0, tile} : Choice{GemmKernel::Library};
}

using Key = std::tuple<int64_t, int64_t, int64_t, int, int, int, int, int>;
std::map<Key, Plan> plans;

hipDataType dataType(DType dt) {
  switch (dt) {
  case DType::F32:
    return HIP_R_32F;
  case DType::F16:
    return HIP_R_16F;
  default:
    return HIP_R_16BF;
  }
}

void destroyPlan(Plan &p) {
  if (p.d) hipblasLtMatrixLayoutDestroy(p.d);
  if (p.b) hipblasLtMatrixLayoutDestroy(p.b);
  if (p.a) hipblasLtMatrixLayoutDestroy(p.a);
  if (p.op) hipblasLtMatmulDescDestroy(p.op);
  p = Plan{};
}

constexpr int kCandidates = 16; // heuristic answers looked through for one that needs no workspace

// Builds (once per shape, flags and type) the library's descriptors and picks its
// algorithms.  No measurement, no allocation beyond the library's host-side descriptors.
Plan &getPlan(DType dt, int64_t M, int64_t N, int64_t K, bool hasBias, int act, bool hasResidual, bool weightKMajor) {
  const bool relu = act == ACT_RELU;
  const Key key{M, N, K, (int)hasBias, act, (int)hasResidual, (int)dt, (int)weightKMajor};
  auto it = plans.find(key);
  if (it != plans.end()) return it->second;

  Plan p;
  const hipDataType t = dataType(dt);
  MGPU_CHECK_BLAS(hipblasLtMatmulDescCreate(&p.op, HIPBLAS_COMPUTE_32F, HIP_R_32F));
  hipblasLtEpilogue_t epilogue = HIPBLASLT_EPILOGUE_DEFAULT;
  if (hasBias && relu)
    epilogue = HIPBLASLT_EPILOGUE_RELU_BIAS;
  else if (hasBias)
    epilogue = HIPBLASLT_EPILOGUE_BIAS;
  else if (relu)
    epilogue = HIPBLASLT_EPILOGUE_RELU;
  MGPU_CHECK_BLAS(hipblasLtMatmulDescSetAttribute(p.op, HIPBLASLT_MATMUL_DESC_EPILOGUE, &epilogue,
                                                  sizeof(epilogue)));
  if (hasBias) {
    const int32_t biasType = (int32_t)t;
    MGPU_CHECK_BLAS(hipblasLtMatmulDescSetAttribute(p.op, HIPBLASLT_MATMUL_DESC_BIAS_DATA_TYPE,
                                                    &biasType, sizeof(biasType)));
  }
  // Column-major view of the row-major operands: A = weight (N x K, ld N; a K-major weight is
  // the K x N matrix with ld K, transposed), B = input (K x M, ld K), C/D = output (N x M, ld N).
  if (weightKMajor) {
    const hipblasOperation_t transposed = HIPBLAS_OP_T;
    MGPU_CHECK_BLAS(hipblasLtMatmulDescSetAttribute(p.op, HIPBLASLT_MATMUL_DESC_TRANSA, &transposed, sizeof(transposed)));
    MGPU_CHECK_BLAS(hipblasLtMatrixLayoutCreate(&p.a, t, K, N, K));
  } else {
    MGPU_CHECK_BLAS(hipblasLtMatrixLayoutCreate(&p.a, t, N, K, N));
  }
  MGPU_CHECK_BLAS(hipblasLtMatrixLayoutCreate(&p.b, t, K, M, K));
  MGPU_CHECK_BLAS(hipblasLtMatrixLayoutCreate(&p.d, t, N, M, N));

  hipblasLtMatmulPreference_t pref = nullptr;
  MGPU_CHECK_BLAS(hipblasLtMatmulPreferenceCreate(&pref));
  const uint64_t ws = workspaceSize;
  MGPU_CHECK_BLAS(hipblasLtMatmulPreferenceSetAttribute(
      pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &ws, sizeof(ws)));
  hipblasLtMatmulHeuristicResult_t results[kCandidates] = {};
  int returned = 0;
  const hipblasStatus_t st = hipblasLtMatmulAlgoGetHeuristic(ltHandle, p.op, p.a, p.b, p.d, p.d,
                                                             pref, kCandidates, results, &returned);
  hipblasLtMatmulPreferenceDestroy(pref);
  if (st != HIPBLAS_STATUS_SUCCESS || returned == 0) {
    destroyPlan(p);
    fail("matmul: hipBLASLt has no algorithm for M=" + std::to_string(M) + " N=" +
         std::to_string(N) + " K=" + std::to_string(K));
  }
  p.algo = results[0].algo;
  p.algoWorkspace = results[0].workspaceSize;
  for (int c = 0; c < returned && !p.hasNoWs; c++)
    if (results[c].state == HIPBLAS_STATUS_SUCCESS && results[c].workspaceSize == 0) {
      p.algoNoWs = results[c].algo;
      p.hasNoWs = true;
    }

  return plans.emplace(key, p).first->second;
}

} // namespace

void gemmInit() {
  if (ltHandle) return;
  MGPU_CHECK_BLAS(hipblasLtCreate(&ltHandle));
}

void gemmDeinit() {
  std::lock_guard<std::mutex> lock(planMutex);
  for (auto &kv : plans) destroyPlan(kv.second);
  plans.clear();
  for (auto &kv : workspaceOf)
    if (kv.second) (void)hipFree(kv.second);
  workspaceOf.clear();
  if (ltHandle) hipblasLtDestroy(ltHandle);
  ltHandle = nullptr;
}

bool gemmPrefersKMajor(DType dt, const void *weight, const void *bias, int64_t M, int64_t N, int64_t K, bool hasBias, int act,
                       bool hasResidual) {
  if (forcedKernel()) return forcedKernel() == 1;
  if (const TableEntry *e = tableRow(dt, M, N, K, hasBias, act, hasResidual)) return e->kMajorLibrary != 0;
  // The library's kernels for K-major weights were ahead of its kernels for [K, N] weights at every shape measured, so the copy
  // pays wherever the library would serve the shape anyway.  Not where a kernel of ours does, which is ahead of the library on the copy
  // too, and whose product may be split, the copy's not (us a layer, gemm_round's and gemm_ksplit's products from copies / as they
  // are: BERT layer of 768 on 6 x 129 tokens 61.8 / 51.2, 32 x 128 95.0 / 92.3, of 512 on 10 x 136 58.9 / 47.4, 77 28.0 / 24.9; decoding
  // layer of 2048, ffn 8192, on 500 123 / 99, of 512 on 2 x 750 67.2 / 59.0; over 820 layers 0.94 of the time on average, 17 of them
  // more than 3 % slower, all of 2048 with an ffn of 2048: on 700 tokens 97 / 104, where gemm_round takes 96 columns and 128 would be
  // ahead, on 93 51 / 53).
  alignas(16) static const char aligned[16] = {};
  return chooseKernel(dt, aligned, weight, hasBias ? bias : nullptr, hasResidual ? aligned : nullptr, aligned, M, N, K, hasBias, act,
                      hasResidual, false).kernel == GemmKernel::Library;
}

int gemmWideWidth(DType dt, int64_t M, int64_t N, int64_t K, int act, bool hasResidual) {
  alignas(16) static const char aligned[16] = {};
  return wideWidth(dt, aligned, aligned, aligned, hasResidual ? aligned : nullptr, aligned, M, N, K, act);
}

GemmKernel gemmKernelFor(DType dt, int64_t M, int64_t N, int64_t K, bool hasBias, int act, bool hasResidual, bool weightKMajor) {
  alignas(16) static const char aligned[16] = {};
  return chooseKernel(dt, aligned, aligned, hasBias ? aligned : nullptr, hasResidual ? aligned : nullptr, aligned, M, N, K, hasBias, act,
                      hasResidual, weightKMajor).kernel;
}

bool gemmWantsKMajorCast(DType dt, int64_t M, int64_t N, int64_t K, bool hasBias, int act, bool hasResidual) {
  // Wherever the [K, N] weight would be the library's, as its kernels for the other layout are ahead, and gemm_ksplit's
  // where it takes that layout of a short reduction.
  if (gemmKernelFor(dt, M, N, K, hasBias, act, hasResidual, false) != GemmKernel::Library) return false;
  return K <= 512 || gemmKernelFor(dt, M, N, K, hasBias, act, hasResidual, true) == GemmKernel::Library;
}

// Splitting pays where a product has so few tiles that most CUs idle behind a long reduction: the layers' projection and
// second FFN product at a few to some 2000 tokens.  Estimates as in chooseKernel, plus what writing the planes and reading
// them in the LayerNorm behind costs over a product and its LayerNorm, fitted to 330 splits (7 % rms for gemm_mfma's, 12 % for
// gemm_ksplit's; us, product + LayerNorm whole / split: 77 x 768 x 3072 11.6 / 8.7, 1024 x 768 x 3072 19.9 / 17.1, 1368 x 768 x
// 3072 23.1 / 18.8).  Where the estimates differ by less than a tenth the product stays whole
// (1024 x 1024 x 2048 16.0 / 15.6): the choice is 1.7 % behind the best over 110 shapes, at worst 8 % behind the whole product.
PartialPlan gemmPartialPlan(const void *in, const void *weight, int64_t M, int64_t N, int64_t K, bool weightKMajor) {
  PartialPlan best;
  if (forcedKernel() || weightKMajor || K < 512) return best;
  const GemmKernel whole = chooseKernel(DType::F16, in, weight, weight, nullptr, weight, M, N, K, true, ACT_NONE, false, false).kernel;
  double bestCost;
  if (whole == GemmKernel::Wide) (void)gemmWideBest(M, N, K, ACT_NONE, false, &bestCost);
  else if (whole == GemmKernel::Round) bestCost = gemmMfmaCost(M, N, (K + 63) / 64 * 64, ACT_NONE);
  else if (whole == GemmKernel::Mfma) bestCost = gemmMfmaCost(M, N, K, ACT_NONE);
  else if (whole == GemmKernel::KSplit) (void)gemmKSplitBest(M, N, K, ACT_NONE, &bestCost);
  else return best;
  bestCost = 0.9 * bestCost;
  const bool mfmaOk = gemmMfmaSupportsRagged(DType::F16, in, weight, nullptr, nullptr, weight, M, N, K);
  const bool kSplitOk = gemmKSplitSupports(DType::F16, in, weight, nullptr, nullptr, weight, M, N, K);
  for (int parts = 2; parts <= 4 && K / parts >= 256; parts++) {
    const double elements = (double)M * (double)N * parts, mfmaPlanes = 2.6e-6 * elements, kSplitPlanes = 0.6 + 1.2e-6 * elements;
    if (mfmaOk && gemmMfmaPartialCost(M, N, K, parts) + mfmaPlanes < bestCost) {
      bestCost = gemmMfmaPartialCost(M, N, K, parts) + mfmaPlanes;
      best = PartialPlan{parts, true, KSplitTile::T32x32};
    }
    double cost;
    const KSplitTile tile = gemmKSplitBest(M, N, K, ACT_NONE, &cost, parts);
    if (kSplitOk && cost + kSplitPlanes < bestCost) {
      bestCost = cost + kSplitPlanes;
      best = PartialPlan{parts, false, tile};
    }
  }
  return best;
}

void gemmPartialF16(const PartialPlan &plan, const void *in, const void *weight, float *planes, int64_t M, int64_t N, int64_t K,
                    hipStream_t stream) {
  if (plan.mfma) gemmMfmaPartialF16(in, weight, planes, M, N, K, plan.parts, stream);
  else gemmKSplitPartialF16(in, weight, planes, M, N, K, plan.tile, plan.parts, stream);
}

bool matmulResidualF32(const void *input, const void *weight, const void *bias, const void *residual, float *output, int64_t M, int64_t N,
                       int64_t K, bool weightKMajor, hipStream_t stream) {
  if (!bias || !residual || !aligned16(output)) return false;
  // (gemm_wide wherever it can go, also on shallow products: its unrounded result saves a pass)
  const int wide = weightKMajor || K % 64 ? 0 : wideWidth(DType::F16, input, weight, bias, residual, output, M, N, K, ACT_NONE);
  if (wide) {
    gemmWideResidualF32(input, weight, bias, residual, output, M, N, K, wide, stream);
    return true;
  }
  const Choice choice = chooseKernel(DType::F16, input, weight, bias, residual, output, M, N, K, true, ACT_NONE, true, weightKMajor);
  if (choice.kernel == GemmKernel::Round) gemmRoundResidualF32(input, weight, bias, residual, output, M, N, K, choice.width, stream);
  else if (choice.kernel == GemmKernel::KSplit) gemmKSplitResidualF32(input, weight, bias, residual, output, M, N, K, choice.tile, weightKMajor, stream);
  else return false;
  return true;
}

void matmulEx(DType dt, const void *input, const void *weight, const void *bias, void *output,
              const void *residual, int64_t M, int64_t N, int64_t K, bool hasBias, int act,
              bool hasResidual, hipStream_t stream, bool weightKMajor) {
  if (M < 0 || N < 0 || K < 0) fail("matmul: negative shape");
  if (M == 0 || N == 0) return;
  if (K == 0) fail("matmul: K must be positive");
  if (!ltHandle) fail("matmul: gpuOpsInit() has not been called");
  if (!input || !weight || !output) fail("matmul: null pointer");
  if (hasBias && !bias) fail("matmul: hasBias set but bias is null");
  if (hasResidual && !residual) fail("matmul: hasResidual set but residual is null");
  if (act < ACT_NONE || act > ACT_GELU) fail("matmul: unknown activation");
  if (act != ACT_NONE && hasResidual)
    fail("matmul: an activation cannot be combined with a residual");

  const void *b = hasBias ? bias : nullptr, *r = hasResidual ? residual : nullptr;
  const Choice choice = chooseKernel(dt, input, weight, b, r, output, M, N, K, hasBias, act, hasResidual, weightKMajor);
  switch (choice.kernel) {
  case GemmKernel::Wide:
    gemmWide(dt, input, weight, b, r, output, M, N, K, act, choice.width, stream);
    return;
  case GemmKernel::Round:
    gemmRound(dt, input, weight, b, r, output, M, N, K, act, choice.width, stream);
    return;
  case GemmKernel::Mfma:
    gemmMfmaRagged(dt, input, weight, b, r, output, M, N, K, act, stream);
    return;
  case GemmKernel::KSplit:
    gemmKSplit(dt, input, weight, b, r, output, M, N, K, act, choice.tile, weightKMajor, stream);
    return;
  case GemmKernel::F32Small:
    gemmF32Small(static_cast<const float *>(input), static_cast<const float *>(weight), static_cast<const float *>(b),
                 static_cast<const float *>(r), static_cast<float *>(output), M, N, K, act, stream);
    return;
  case GemmKernel::Library:
    break;
  }
  std::lock_guard<std::mutex> lock(planMutex);
  const Plan &p = getPlan(dt, M, N, K, hasBias, act, hasResidual, weightKMajor);
  if (hasBias)
    MGPU_CHECK_BLAS(hipblasLtMatmulDescSetAttribute(p.op, HIPBLASLT_MATMUL_DESC_BIAS_POINTER, &bias,
                                                    sizeof(bias)));
  const float alpha = 1.0f, beta = hasResidual ? 1.0f : 0.0f;
  // The stream's own workspace; a stream first met under capture has none and runs the
  // first algorithm that does without.
  void *workspace = p.algoWorkspace ? workspaceFor(stream) : nullptr;
  const hipblasLtMatmulAlgo_t *algo = &p.algo;
  if (p.algoWorkspace && !workspace) {
    if (!p.hasNoWs) fail("matmul: the library needs a workspace for this shape and none could be allocated now (stream capture or out of memory); run it once on this stream before capturing");
    algo = &p.algoNoWs;
  }
  MGPU_CHECK_BLAS(hipblasLtMatmul(ltHandle, p.op, &alpha, weight, p.a, input, p.b, &beta,
                                  hasResidual ? residual : output, p.d, output, p.d, algo,
                                  workspace, workspace ? workspaceSize : 0, stream));
  if (act == ACT_GELU) {
    if (dt == DType::F16)
      geluInPlaceF16(output, (size_t)M * N, stream);
    else if (dt == DType::BF16)
      geluInPlaceBF16(output, (size_t)M * N, stream);
    else
      geluInPlaceF32(static_cast<float *>(output), (size_t)M * N, stream);
  }
}

} // namespace mgpu
