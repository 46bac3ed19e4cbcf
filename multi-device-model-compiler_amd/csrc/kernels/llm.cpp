// Transformer layers composed from the kernels of this library.
//
// decodingContextLayer is the counterpart of mgpuLLMDecodingContextLayer
// (lib/Kernels/GPU/LLM.cu:26-159): fp32 tensors in and out, fp16 compute.
// Kept from the reference: the dataflow (pre-LN, gamma = 1 / beta = 0
// LayerNorms at eps 1e-5, packed-QKV attention, bias epilogues, residual
// through the GEMM's C operand).  Changed on purpose:
//  * head_num, norm_first, is_casual and is_relu are honoured (the reference
//    ignores them and runs 8 heads x 128, pre-LN, causal, ReLU:
//    LLM.cu:18-19,79-81,119-121); norm_first = false is the post-LN ordering
//    of the same blocks;
//  * one arena instead of 12 allocations and frees per call, and the arena is
//    kept per caller stream between calls (an allocation and a free per call
//    cost 14 us of host time, about a tenth of a BERT-base layer): it grows to
//    the largest layer that stream has run and is returned by gpuLLMOpsDeinit.
//    Calls on one stream are ordered by the stream; calls on different streams
//    get different arenas (and, with the weight cache on, side streams).  A call made under stream
//    capture never touches the kept arena: it allocates and frees inside the
//    capture, so the graph owns its temporaries and a later eager call that
//    grows (frees and replaces) the stream's arena cannot pull memory from
//    under a graph that is still replayed;
//  * one kernel casts all seven weight and bias arrays and the input, with its LayerNorm where that comes first, on the caller's stream
//    (the reference casts each on a side stream; here the casts are bound by
//    memory, so beside a GEMM they only slow it, and their launches and events
//    were half of the host time of a small layer: 4096 x 2048 321 -> 289 us,
//    240 x 768 112 -> 47 us); it writes K-major the weights whose GEMM is the
//    library's, which has faster kernels for that layout.  The gamma = 1 /
//    beta = 0 vectors are written once per model width, not per call;
//  * the final fp16 -> fp32 cast is the last GEMM's or LayerNorm's epilogue, and a kernel behind it only where that has none
//    (the reference issues it on the side stream without waiting for that GEMM: LLM.cu:136-141).
//
// bertEncoderLayerF16 is the post-LN BERT encoder layer on fp16 tensors (GELU,
// learned LayerNorm affine, optional key-padding lengths); the reference has
// no such entry point.
#include "common.hpp"

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <tuple>
#include "mgpu_ops_internal.hpp"

namespace mgpu {

namespace {

bool initialised = false;
constexpr int kGemms = 4; // of a layer

// What the layers keep per caller stream between calls: the arena and, for the
// weight cache's conversions, a side stream with its fork event (two caller streams
// in flight at once must not re-record one another's event).
struct StreamState {
  void *base = nullptr; // arena
  size_t bytes = 0;
  hipStream_t side = nullptr;
  hipEvent_t forkEvent = nullptr;
};
std::mutex scratchMutex;
std::map<hipStream_t, StreamState> stateOf;

bool isCapturing(hipStream_t s) {
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(s, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone;
}

// The caller stream's state, with its side stream and event in place.  They
// are created on the stream's first call that asks the weight cache; scratchMutex must be held.
StreamState &sideOf(hipStream_t s) {
  StreamState &st = stateOf[s];
  if (!st.side) {
    MGPU_CHECK_HIP(hipStreamCreateWithFlags(&st.side, hipStreamNonBlocking));
    MGPU_CHECK_HIP(hipEventCreateWithFlags(&st.forkEvent, hipEventDisableTiming));
  }
  return st;
}

// Opt-in cache of the reference layer's weights in fp16 (mgpuLLMOpsCacheWeights).  The layer's
// ABI hands it fp32 weights and the reference casts all of them on every call (LLM.cu:55-57,
// 84-90,100-106,124-130): 300 MB of HBM traffic per call at d_model 2048, on a side stream, next
// to the GEMMs.  With the cache on, an array is cast the first time its (address, shape) is seen
// and the fp16 copy is kept until the cache is switched off or gpuLLMOpsDeinit; the caller
// promises not to change a cached array in place.  The layout of a copy is the cache's own
// business: where gemmPrefersKMajor says so for the GEMM that reads it - where the library would serve it, with N or K no multiple
// of 8 - a weight matrix is stored transposed, [N, K] with K contiguous, for which the library's kernels are faster (4096 x 2304 x
// 768: 19 against 29 us).  The BERT layer, whose weights arrive in fp16, takes only such transposed copies from the cache.  Off by
// default: per-call casts, as in
// the reference.  Guarded by scratchMutex.
bool weightCacheOn = false;
struct CachedWeight {
  void *half = nullptr;
  hipEvent_t ready = nullptr; // recorded behind the conversion that filled the copy
  bool done = false;          // the event has been seen complete: nobody needs to wait for it any more
  // What a stream that is about to read the copy has to wait for (nothing, once the conversion
  // has finished: a wait on a complete event still costs the stream a barrier packet).
  hipEvent_t pending() {
    if (!done) {
      if (hipEventQuery(ready) == hipSuccess) done = true;
      else (void)hipGetLastError(); // "not ready" is an answer, not an error the next launch check should find
    }
    return done ? nullptr : ready;
  }
};
// (array, rows, columns - 0 for a vector -, stored K-major?)
using WeightKey = std::tuple<const void *, int64_t, int64_t, bool>;
std::map<WeightKey, CachedWeight> weightCache;

// The cache's copy of a weight or bias array, made now - on `convert`, behind whatever that
// stream already holds - if this is the first sight of it.  fp32 arrays are cast to fp16; a matrix
// asked for K-major is stored transposed.  scratchMutex held; not under stream capture.
CachedWeight &cachedWeight(const void *src, bool srcIsF32, int64_t rows, int64_t cols, bool kMajor,
                                 hipStream_t convert) {
  const WeightKey key{src, rows, cols, kMajor};
  auto hit = weightCache.find(key);
  if (hit != weightCache.end()) return hit->second;
  const int64_t elems = cols ? rows * cols : rows;
  CachedWeight fresh; // entered into the cache only once its conversion is queued
  MGPU_CHECK_HIP(hipMalloc(&fresh.half, (size_t)elems * 2));
  try {
    MGPU_CHECK_HIP(hipEventCreateWithFlags(&fresh.ready, hipEventDisableTiming));
    if (srcIsF32 && kMajor) transposeCastF32ToF16(fresh.half, static_cast<const float *>(src), rows, cols, convert);
    else if (srcIsF32) castF32ToF16(fresh.half, static_cast<const float *>(src), elems, convert);
    else if (kMajor) transpose16(fresh.half, src, rows, cols, convert);
    else fail("weight cache: nothing to convert");
    MGPU_CHECK_HIP(hipEventRecord(fresh.ready, convert));
  } catch (...) {
    if (fresh.ready) (void)hipEventDestroy(fresh.ready);
    (void)hipFree(fresh.half);
    throw;
  }
  return weightCache.emplace(key, fresh).first->second;
}

bool cacheIsOn() {
  std::lock_guard<std::mutex> lock(scratchMutex);
  return weightCacheOn;
}

void dropWeightCache() { // scratchMutex held; the device idle or the copies no longer in use
  for (auto &kv : weightCache) {
    if (kv.second.half) (void)hipFree(kv.second.half);
    if (kv.second.ready) (void)hipEventDestroy(kv.second.ready);
  }
  weightCache.clear();
}

// gamma = 1, beta = 0 in fp16 for the reference layer's LayerNorms, one pair
// per model width, written once and kept until gpuLLMOpsDeinit.
struct Identity {
  void *gamma = nullptr, *beta = nullptr;
};
std::map<int64_t, Identity> identityOf;

// Null when the pair does not exist yet and cannot be made now (stream capture).
const Identity *identityAffine(int64_t d, hipStream_t stream) {
  std::lock_guard<std::mutex> lock(scratchMutex);
  auto it = identityOf.find(d);
  if (it != identityOf.end()) return &it->second;
  if (isCapturing(stream)) return nullptr;
  Identity id;
  MGPU_CHECK_HIP(hipMalloc(&id.gamma, (size_t)d * 2));
  MGPU_CHECK_HIP(hipMalloc(&id.beta, (size_t)d * 2));
  fillF16(id.gamma, d, 1.0f, stream);
  fillF16(id.beta, d, 0.0f, stream);
  MGPU_CHECK_HIP(hipStreamSynchronize(stream)); // once per width: any stream may read the pair from now on
  return &identityOf.emplace(d, id).first->second;
}

// Bump allocator over one stream-ordered allocation; every slice is 256-byte
// aligned so all vectorised kernels see aligned pointers.
class Arena {
public:
  size_t reserve(size_t bytes) {
    const size_t at = total_;
    total_ += (bytes + 255) & ~size_t(255);
    return at;
  }
  // Memory usable by work enqueued on `s` from here on.
  void allocate(hipStream_t s) {
    const size_t need = total_ ? total_ : 256;
    if (isCapturing(s)) { // the graph owns its temporaries: allocated and freed inside the capture
      MGPU_CHECK_HIP(hipMallocAsync(&base_, need, s));
      perCall_ = true;
      return;
    }
    std::lock_guard<std::mutex> lock(scratchMutex);
    StreamState &kept = stateOf[s];
    if (kept.bytes >= need) {
      base_ = kept.base;
      return;
    }
    if (kept.base) MGPU_CHECK_HIP(hipFreeAsync(kept.base, s)); // after the work already queued on s
    kept.base = nullptr;
    kept.bytes = 0;
    MGPU_CHECK_HIP(hipMallocAsync(&base_, need, s));
    kept.base = base_;
    kept.bytes = need;
  }
  void release(hipStream_t s) {
    if (base_ && perCall_) MGPU_CHECK_HIP(hipFreeAsync(base_, s));
    base_ = nullptr;
  }
  template <typename T = void> T *at(size_t offset) const {
    return reinterpret_cast<T *>(static_cast<char *>(base_) + offset);
  }

private:
  void *base_ = nullptr;
  size_t total_ = 0;
  bool perCall_ = false;
};

} // namespace

void llmInit() { initialised = true; }

void llmDeinit() {
  std::lock_guard<std::mutex> lock(scratchMutex);
  if (!stateOf.empty()) (void)hipDeviceSynchronize(); // the streams the arenas were ordered on may be gone
  for (auto &kv : stateOf) {
    StreamState &st = kv.second;
    if (st.base) (void)hipFreeAsync(st.base, nullptr);
    if (st.side) (void)hipStreamDestroy(st.side);
    if (st.forkEvent) (void)hipEventDestroy(st.forkEvent);
  }
  if (!stateOf.empty()) (void)hipStreamSynchronize(nullptr);
  stateOf.clear();
  for (auto &kv : identityOf) {
    if (kv.second.gamma) (void)hipFree(kv.second.gamma);
    if (kv.second.beta) (void)hipFree(kv.second.beta);
  }
  identityOf.clear();
  dropWeightCache();
  weightCacheOn = false;
  initialised = false;
}

void llmCacheWeights(bool enable) {
  std::lock_guard<std::mutex> lock(scratchMutex);
  if (!enable && !weightCache.empty()) {
    (void)hipDeviceSynchronize(); // a layer in flight may still read the copies
    dropWeightCache();
  }
  weightCacheOn = enable;
}

void decodingContextLayer(float *input, float *qkv, float *gemm_weight, float *gemm_bias,
                          float *ffn1_weight, float *ffn1_bias, float *ffn2_weight,
                          float *ffn2_bias, float *output, int64_t batch, int64_t seq_len,
                          int64_t d_model, int64_t ffn, int64_t heads, bool norm_first,
                          bool causal, bool relu, hipStream_t stream) {
  if (!initialised) fail("mgpuLLMDecodingContextLayer: gpuOpsInit() has not been called");
  if (batch < 0 || seq_len < 0 || d_model <= 0 || ffn <= 0 || heads <= 0)
    fail("mgpuLLMDecodingContextLayer: bad shape");
  if (d_model % heads || d_model / heads < 8 || d_model / heads > 256 || (d_model / heads) % 8)
    fail("mgpuLLMDecodingContextLayer: d_model / head_num must be a multiple of 8 between 8 and 256");
  if (batch == 0 || seq_len == 0) return;
  if (!input || !qkv || !gemm_weight || !gemm_bias || !ffn1_weight || !ffn1_bias || !ffn2_weight ||
      !ffn2_bias || !output)
    fail("mgpuLLMDecodingContextLayer: null pointer");
  const int64_t M = batch * seq_len, d = d_model;
  if (M > 0x7fffffff || d > 0x7fffffff) fail("mgpuLLMDecodingContextLayer: shape too large");
  constexpr size_t h = 2; // bytes per fp16

  Arena arena;
  const size_t oX = arena.reserve(M * d * h), oLn = arena.reserve(M * d * h);
  const size_t oGamma = arena.reserve(d * h), oBeta = arena.reserve(d * h);
  const size_t oWqkv = arena.reserve(d * 3 * d * h), oQkv = arena.reserve(M * 3 * d * h);
  const size_t oWo = arena.reserve(d * d * h), oBo = arena.reserve(d * h);
  const size_t oProj = arena.reserve(M * d * h), oY = arena.reserve(M * d * h);
  const size_t oW1 = arena.reserve(d * ffn * h), oB1 = arena.reserve(ffn * h);
  const size_t oF = arena.reserve(M * ffn * h);
  const size_t oW2 = arena.reserve(ffn * d * h), oB2 = arena.reserve(d * h);
  const size_t oOut = arena.reserve(M * d * h);
  const int act = relu ? ACT_RELU : ACT_GELU;
  const bool useCache = cacheIsOn() && !isCapturing(stream); // a capture neither allocates nor reads the cache's events
  bool kMajor[kGemms]; // GEMM g gets a transposed copy of its weight
  {
    // (the copies, in the cache or in the arena, are aligned)
    auto prefers = [&](int64_t n, int64_t k, bool bias, int activation, bool residual) {
      return useCache ? gemmPrefersKMajor(DType::F16, nullptr, nullptr, M, n, k, bias, activation, residual)
                      : gemmWantsKMajorCast(DType::F16, M, n, k, bias, activation, residual);
    };
    kMajor[0] = prefers(3 * d, d, false, ACT_NONE, false);
    kMajor[1] = prefers(d, d, true, ACT_NONE, false);
    kMajor[2] = prefers(ffn, d, true, act, false);
    kMajor[3] = prefers(d, ffn, true, ACT_NONE, norm_first);
  }
  // (the operands of both split products are slices of the arena: aligned)
  const bool sumsOk = partialSumsSupports(nullptr, nullptr, nullptr, nullptr, output, M, d);
  const PartialPlan projPlan = sumsOk ? gemmPartialPlan(nullptr, nullptr, M, d, d, kMajor[1]) : PartialPlan{};
  const PartialPlan ffn2Plan = sumsOk ? gemmPartialPlan(nullptr, nullptr, M, d, ffn, kMajor[3]) : PartialPlan{};
  const size_t oPlanes = arena.reserve((size_t)std::max(projPlan.parts, ffn2Plan.parts) * M * d * 4);

  arena.allocate(stream);
  // The seven weight and bias arrays in fp16: cast now, all in one launch, or - with the weight cache
  // on - taken from the cache (cast once, when first seen, on a side stream).
  struct Operand {
    const float *src;
    int64_t rows, cols; // [K, N] of a weight; a bias is rows elements and cols = 0
    size_t slot;        // where the per-call copy goes in the arena
    int group;          // the GEMM (0..3) that reads it
    void *half;         // the fp16 copy the GEMM is given
  };
  Operand ops[7] = {{qkv, d, 3 * d, oWqkv, 0, nullptr},      {gemm_weight, d, d, oWo, 1, nullptr},
                    {gemm_bias, d, 0, oBo, 1, nullptr},      {ffn1_weight, d, ffn, oW1, 2, nullptr},
                    {ffn1_bias, ffn, 0, oB1, 2, nullptr},    {ffn2_weight, ffn, d, oW2, 3, nullptr},
                    {ffn2_bias, d, 0, oB2, 3, nullptr}};
  hipEvent_t cachedReady[7] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
  if (useCache) {
    // (an array's first conversion runs on the side stream, behind what already sits on `stream`)
    std::lock_guard<std::mutex> lock(scratchMutex);
    const StreamState &st = sideOf(stream);
    bool forked = false;
    for (int i = 0; i < 7; i++) {
      Operand &op = ops[i];
      const bool transposed = op.cols && kMajor[op.group];
      if (!forked && !weightCache.count(WeightKey{op.src, op.rows, op.cols, transposed})) {
        MGPU_CHECK_HIP(hipEventRecord(st.forkEvent, stream));
        MGPU_CHECK_HIP(hipStreamWaitEvent(st.side, st.forkEvent, 0));
        forked = true;
      }
      CachedWeight &cw = cachedWeight(op.src, true, op.rows, op.cols, transposed, st.side);
      op.half = cw.half;
      cachedReady[i] = cw.pending();
    }
  } else {
    for (Operand &op : ops) op.half = arena.at(op.slot);
  }
  auto join = [&](int group) {
    for (int i = 0; i < 7; i++)
      if (ops[i].group == group && cachedReady[i]) MGPU_CHECK_HIP(hipStreamWaitEvent(stream, cachedReady[i], 0));
  };
  const void *wqkvH = ops[0].half, *woH = ops[1].half, *boH = ops[2].half, *w1H = ops[3].half, *b1H = ops[4].half,
             *w2H = ops[5].half, *b2H = ops[6].half;

  const void *gamma = arena.at(oGamma), *beta = arena.at(oBeta);
  if (const Identity *id = identityAffine(d, stream)) {
    gamma = id->gamma;
    beta = id->beta;
  } else { // under capture, first use of this width: the pair lives in the arena
    fillF16(arena.at(oGamma), d, 1.0f, stream);
    fillF16(arena.at(oBeta), d, 0.0f, stream);
  }

  // The casts: the weights' and, in the same launch, the input's - with its LayerNorm where that comes first and the width allows
  // (fp16 copy of the input, the residual of the second LayerNorm, and its LayerNorm: one kernel where the width allows, else the
  // reference's two).
  {
    CastJob jobs[8];
    int count = 0;
    if (!useCache)
      for (const Operand &op : ops) jobs[count++] = CastJob{op.src, op.half, op.rows, op.cols ? op.cols : 1, op.cols && kMajor[op.group], false};
    const bool fused = norm_first && (count ? castWeightsLayerNormF32ToF16(jobs, count, input, gamma, beta, arena.at(oX), arena.at(oLn), 1e-5f, (int)M, (int)d, stream)
                                            : castLayerNormF32ToF16(input, gamma, beta, arena.at(oX), arena.at(oLn), 1e-5f, (int)M, (int)d, stream));
    if (!fused) {
      jobs[count++] = CastJob{input, arena.at(oX), M, d, false, false};
      castWeightsF32ToF16(jobs, count, stream);
      if (norm_first) layerNorm(DType::F16, arena.at(oX), nullptr, gamma, beta, nullptr, arena.at(oLn), 1e-5f, (int)M, (int)d, stream);
    }
  }

  // LN(in . w + bias + residual), the rounded sum to sumOut when it is not null.  Where the sum is wanted and gemm_wide serves the
  // product, its epilogue adds the residual and rounds the sum once, and the LayerNorm reads and writes one matrix each instead of two
  // (4096 x 2048 x 2048, product + LayerNorm 39.0 + 14.5 -> 42.2 + 6.8 us).  Mean and variance then come from the rounded sum, as the
  // normalised value does either way; the kernel that adds the residual itself takes them from the fp32 sum of the rounded product.
  auto productAddNorm = [&](const PartialPlan &plan, const void *in, const void *w, const void *bias, int64_t K, bool transposed,
                            const void *residual, void *sumOut, void *out) {
    if (plan.parts) {
      gemmPartialF16(plan, in, w, arena.at<float>(oPlanes), M, d, K, stream);
      partialSumsLayerNormF16(arena.at<float>(oPlanes), plan.parts, bias, residual, gamma, beta, sumOut, out, 1e-5f, M, d, stream);
      return;
    }
    if (sumOut && !transposed && gemmWideWidth(DType::F16, M, d, K, ACT_NONE, true)) {
      matmulEx(DType::F16, in, w, bias, sumOut, residual, M, d, K, true, ACT_NONE, true, stream, false);
      layerNorm(DType::F16, sumOut, nullptr, gamma, beta, nullptr, out, 1e-5f, (int)M, (int)d, stream);
      return;
    }
    matmulEx(DType::F16, in, w, bias, arena.at(oProj), nullptr, M, d, K, true, ACT_NONE, false, stream, transposed);
    layerNorm(DType::F16, arena.at(oProj), residual, gamma, beta, sumOut, out, 1e-5f, (int)M, (int)d, stream);
  };

  if (norm_first) {
    // y = x + proj(attention(LN(x))), out = y + ffn(LN(y))
    join(0);
    matmulEx(DType::F16, arena.at(oLn), wqkvH, nullptr, arena.at(oQkv), nullptr, M, 3 * d,
             d, false, ACT_NONE, false, stream, kMajor[0]);

    // Attention context overwrites the first LayerNorm output, like the reference.
    fusedMHA(DType::F16, arena.at(oQkv), nullptr, arena.at(oLn), (int)batch, (int)seq_len,
             (int)heads, (int)(d_model / heads), 1.0f / sqrtf((float)(d_model / heads)), causal, stream);

    join(1);
    productAddNorm(projPlan, arena.at(oLn), woH, boH, d, kMajor[1], arena.at(oX), arena.at(oY), arena.at(oLn));

    join(2);
    matmulEx(DType::F16, arena.at(oLn), w1H, b1H, arena.at(oF), nullptr, M, ffn,
             d, true, relu ? ACT_RELU : ACT_GELU, false, stream, kMajor[2]);

    join(3);
    if (ffn2Plan.parts) { // the fp32 result straight from the sums
      gemmPartialF16(ffn2Plan, arena.at(oF), w2H, arena.at<float>(oPlanes), M, d, ffn, stream);
      partialSumsF32(arena.at<float>(oPlanes), ffn2Plan.parts, b2H, arena.at(oY), output, M, d, stream);
      arena.release(stream);
      return;
    }
    // (or from the product's accumulators: 4096 x 2048 x 2048 42.2 + 11.2 for the cast behind it -> 40.5 us)
    if (matmulResidualF32(arena.at(oF), w2H, b2H, arena.at(oY), output, M, d, ffn, kMajor[3], stream)) {
      arena.release(stream);
      return;
    }
    matmulEx(DType::F16, arena.at(oF), w2H, b2H, arena.at(oOut), arena.at(oY), M,
             d, ffn, true, ACT_NONE, true, stream, kMajor[3]);
  } else {
    // norm_first = false, the post-LN ordering of the same blocks (the reference declares the
    // flag, Ops.h:43-48, and never reads it):  h = LN(x + proj(attention(x))),
    // out = LN(h + ffn(h)), both LayerNorms with gamma = 1 / beta = 0 at eps 1e-5 like the
    // pre-LN ones, every intermediate stored in fp16 where the pre-LN path stores it.
    join(0);
    matmulEx(DType::F16, arena.at(oX), wqkvH, nullptr, arena.at(oQkv), nullptr, M, 3 * d,
             d, false, ACT_NONE, false, stream, kMajor[0]);
    fusedMHA(DType::F16, arena.at(oQkv), nullptr, arena.at(oLn), (int)batch, (int)seq_len,
             (int)heads, (int)(d_model / heads), 1.0f / sqrtf((float)(d_model / heads)), causal, stream);
    join(1);
    // h (in oY) = LN(proj + x); the rounded sum is not needed again
    productAddNorm(projPlan, arena.at(oLn), woH, boH, d, kMajor[1], arena.at(oX), nullptr, arena.at(oY));
    join(2);
    matmulEx(DType::F16, arena.at(oY), w1H, b1H, arena.at(oF), nullptr, M, ffn,
             d, true, relu ? ACT_RELU : ACT_GELU, false, stream, kMajor[2]);
    join(3);
    if (ffn2Plan.parts) { // the fp32 result straight from the LayerNorm (a launch of nine: 40 tokens of 512 36.2 -> 33.7 us)
      gemmPartialF16(ffn2Plan, arena.at(oF), w2H, arena.at<float>(oPlanes), M, d, ffn, stream);
      partialSumsLayerNormF32(arena.at<float>(oPlanes), ffn2Plan.parts, b2H, arena.at(oY), gamma, beta, output, 1e-5f, M, d, stream);
      arena.release(stream);
      return;
    }
    matmulEx(DType::F16, arena.at(oF), w2H, b2H, arena.at(oProj), nullptr, M, d, ffn, true, ACT_NONE, false, stream, kMajor[3]);
    if (layerNormF16ToF32(arena.at(oProj), arena.at(oY), gamma, beta, output, 1e-5f, (int)M, (int)d, stream)) {
      arena.release(stream);
      return;
    }
    layerNorm(DType::F16, arena.at(oProj), arena.at(oY), gamma, beta, nullptr, arena.at(oOut), 1e-5f, (int)M, (int)d, stream);
  }

  castF16ToF32(output, arena.at(oOut), M * d, stream);
  arena.release(stream);
}

void bertEncoderLayerF16(const void *x, const void *wqkv, const void *bqkv, const void *wo,
                         const void *bo, const void *gamma1, const void *beta1, const void *w1,
                         const void *b1, const void *w2, const void *b2, const void *gamma2,
                         const void *beta2, const int32_t *seqlens, void *out, int64_t B,
                         int64_t S, int64_t d, int64_t ffn, int64_t H, float eps,
                         hipStream_t stream) {
  if (B < 0 || S < 0 || d <= 0 || ffn <= 0 || H <= 0) fail("mgpuBertEncoderLayerF16: bad shape");
  if (d % H || d / H < 8 || d / H > 256 || (d / H) % 8)
    fail("mgpuBertEncoderLayerF16: d_model / head_num must be a multiple of 8 between 8 and 256");
  if (B == 0 || S == 0) return;
  if (!x || !wqkv || !bqkv || !wo || !bo || !gamma1 || !beta1 || !w1 || !b1 || !w2 || !b2 ||
      !gamma2 || !beta2 || !out)
    fail("mgpuBertEncoderLayerF16: null pointer");
  const int64_t M = B * S;
  if (M > 0x7fffffff) fail("mgpuBertEncoderLayerF16: shape too large");
  constexpr size_t h = 2;

  Arena arena;
  const size_t oQkv = arena.reserve(M * 3 * d * h), oCtx = arena.reserve(M * d * h);
  const size_t oProj = arena.reserve(M * d * h);
  const size_t oH1 = arena.reserve(M * d * h), oF = arena.reserve(M * ffn * h);
  // The products before the two LayerNorms, split over blocks where few tiles leave CUs idle.  (The weight cache's K-major
  // copies are for the library: such a product stays whole.  The inputs are slices of the arena: aligned.)
  const bool cached = cacheIsOn() && !isCapturing(stream);
  auto planOf = [&](const void *w, const void *bias, const void *residual, const void *gamma, const void *beta, const void *to, int64_t K) {
    if (!partialSumsSupports(bias, residual, gamma, beta, to, M, d)) return PartialPlan{};
    return gemmPartialPlan(nullptr, w, M, d, K, cached && gemmPrefersKMajor(DType::F16, w, bias, M, d, K, true, ACT_NONE, false));
  };
  const PartialPlan projPlan = planOf(wo, bo, x, gamma1, beta1, nullptr, d), ffn2Plan = planOf(w2, b2, nullptr, gamma2, beta2, out, ffn);
  const size_t oPlanes = arena.reserve((size_t)std::max(projPlan.parts, ffn2Plan.parts) * M * d * 4);
  arena.allocate(stream);

  // With the weight cache on, a GEMM for which the library on a K-major weight is the fastest
  // choice gets the cache's transposed copy of its weight (made on this stream at first sight).
  struct Weight {
    const void *w;
    bool kMajor;
  };
  Weight wq{wqkv, false}, wp{wo, false}, wf1{w1, false}, wf2{w2, false};
  {
    std::lock_guard<std::mutex> lock(scratchMutex);
    if (weightCacheOn && !isCapturing(stream)) {
      auto fromCache = [&](Weight &w, const void *bias, int64_t K, int64_t N, int act) {
        if (!gemmPrefersKMajor(DType::F16, w.w, bias, M, N, K, true, act, false)) return;
        CachedWeight &cw = cachedWeight(w.w, false, K, N, true, stream);
        if (hipEvent_t e = cw.pending()) MGPU_CHECK_HIP(hipStreamWaitEvent(stream, e, 0)); // (filled by another stream, perhaps)
        w = Weight{cw.half, true};
      };
      fromCache(wq, bqkv, d, 3 * d, ACT_NONE);
      fromCache(wp, bo, d, d, ACT_NONE);
      fromCache(wf1, b1, d, ffn, ACT_GELU);
      fromCache(wf2, b2, ffn, d, ACT_NONE);
    }
  }

  matmulEx(DType::F16, x, wq.w, bqkv, arena.at(oQkv), nullptr, M, 3 * d, d, true, ACT_NONE, false, stream, wq.kMajor);
  fusedMHA(DType::F16, arena.at(oQkv), seqlens, arena.at(oCtx), (int)B, (int)S, (int)H, (int)(d / H),
           1.0f / sqrtf((float)(d / H)), false, stream);
  // (nobody reads the rounded sums of this layer: they are not written)
  auto productAddNorm = [&](const PartialPlan &plan, const void *in, const Weight &w, const void *bias, int64_t K, const void *residual,
                            const void *gamma, const void *beta, void *to) {
    if (plan.parts && !w.kMajor) {
      gemmPartialF16(plan, in, w.w, arena.at<float>(oPlanes), M, d, K, stream);
      partialSumsLayerNormF16(arena.at<float>(oPlanes), plan.parts, bias, residual, gamma, beta, nullptr, to, eps, M, d, stream);
      return;
    }
    matmulEx(DType::F16, in, w.w, bias, arena.at(oProj), nullptr, M, d, K, true, ACT_NONE, false, stream, w.kMajor);
    layerNorm(DType::F16, arena.at(oProj), residual, gamma, beta, nullptr, to, eps, (int)M, (int)d, stream);
  };
  productAddNorm(projPlan, arena.at(oCtx), wp, bo, d, x, gamma1, beta1, arena.at(oH1));
  matmulEx(DType::F16, arena.at(oH1), wf1.w, b1, arena.at(oF), nullptr, M, ffn, d, true, ACT_GELU, false, stream,
           wf1.kMajor);
  productAddNorm(ffn2Plan, arena.at(oF), wf2, b2, ffn, arena.at(oH1), gamma2, beta2, out);
  arena.release(stream);
}

} // namespace mgpu
