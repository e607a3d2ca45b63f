// The vendor library's matrix product (hipBLASLt) behind the interface of lev_linear_mfma, for prompt-sized row counts:
//   y = act(a . w^T + bias) (+ residual),  a [M, K] bf16 (row stride lda), w [N, K] bf16, y [M, N] bf16 or f32.
// The reference leaves every matrix product to its compiler's library; here the library takes the large tiles
// (hundreds to thousands of rows), where its tuned kernels are ahead of gemm_tile_kernel on most shapes, and only
// with epilogues it has itself: bias, the tanh GELU ("gelu_new"), ReLU, and the residual as the C operand with beta = 1.
// Everything else (other activations, shapes it has no kernel for) returns LEV_LIBRARY_UNSUPPORTED and the caller
// runs the hand-written kernel. Which of the library's kernels runs a shape is not left to its heuristic alone: for
// 256 rows and more the heuristic's candidates are timed once (its first choice is up to twice slower than its best on row
// counts that are no multiple of the tile, 2,052 rows for instance); the other row counts up to the same multiple of 64 try
// only that kernel against the heuristic's first, where that cannot change the result. In the library's column-major terms the row-major problem is
//   D^T [N x M] = w_cm^T [N x K] . a_cm [K x M]  (+ C^T),  with w_cm = w seen as K x N (ld K), a_cm = a seen as K x M (ld lda),
// so that the bias, one value per row of D^T, is the per-output-column bias of the row-major result.
#include <hipblaslt/hipblaslt.h>
#include <hipblaslt/hipblaslt-ext.hpp>
#include <algorithm>
#include <chrono>

#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "common.h"

#define LEV_LIBRARY_UNSUPPORTED 1
#define LEV_LIB_MAX_DEVICES 64
#define LEV_LIB_CANDIDATES 16    // kernels asked of the heuristic for one shape
#define LEV_LIB_TUNE_MIN_ROWS 256  // below, a product is bound by reading its weight and a timing loop over one weight
                                   // (which then sits in the last-level cache) says nothing about the real step
#define LEV_LIB_TUNE_RUNS 4
#define LEV_LIB_ROW_BUCKET 64      // row counts up to the same multiple of this share one timing

namespace {

struct Plan {
  hipblasLtMatmulDesc_t desc = nullptr;
  hipblasLtMatrixLayout_t lw = nullptr, la = nullptr, lc = nullptr, ld = nullptr;
  hipblasLtMatmulAlgo_t algo;
  size_t workspace = 0;
  bool ok = false;
  bool timed = false;  // the candidates have been timed on this shape and algo is the fastest of them
  std::vector<hipblasLtMatmulHeuristicResult_t> candidates;  // in the heuristic's order; algo starts as the first
};

// (device, M, N, K, lda, ldr, ldo, epilogue, output dtype, residual?)
typedef std::tuple<int, int, int, int, long, long, long, int, int, int> PlanKey;

std::mutex g_mutex;
hipblasLtHandle_t g_handle[LEV_LIB_MAX_DEVICES];
std::map<PlanKey, Plan> g_plans;
// What timing chose, by PlanKey with the row count replaced by its bucket (rows_bucket): the library's index of the kernel, the row count it was timed at, and
// the indices of all kernels that add up in the same order there. Row counts of one bucket share it, so a serving run whose steps differ by a few rows times once, not once a row count.
struct Kept {
  int index = -1, rows = 0;
  std::vector<int> order;
};
std::map<PlanKey, Kept> g_kept;

int rows_bucket(int M) { return (M + LEV_LIB_ROW_BUCKET - 1) / LEV_LIB_ROW_BUCKET; }

const char* status_name(hipblasStatus_t s) {
  switch (s) {
    case HIPBLAS_STATUS_SUCCESS: return "success";
    case HIPBLAS_STATUS_NOT_INITIALIZED: return "not initialized";
    case HIPBLAS_STATUS_ALLOC_FAILED: return "allocation failed";
    case HIPBLAS_STATUS_INVALID_VALUE: return "invalid value";
    case HIPBLAS_STATUS_NOT_SUPPORTED: return "not supported";
    case HIPBLAS_STATUS_EXECUTION_FAILED: return "execution failed";
    default: return "error";
  }
}

#define LIB_CHECK(call)                                                                                         \
  do {                                                                                                          \
    hipblasStatus_t s_ = (call);                                                                                \
    if (s_ != HIPBLAS_STATUS_SUCCESS) return lev_fail("linear (library): %s: %s", #call, status_name(s_));       \
  } while (0)

int epilogue_of(int act, bool bias, uint32_t* out) {
  if (act == LEV_ACT_NONE) *out = bias ? HIPBLASLT_EPILOGUE_BIAS : HIPBLASLT_EPILOGUE_DEFAULT;
  else if (act == LEV_ACT_GELU_TANH) *out = bias ? HIPBLASLT_EPILOGUE_GELU_BIAS : HIPBLASLT_EPILOGUE_GELU;
  else if (act == LEV_ACT_RELU) *out = bias ? HIPBLASLT_EPILOGUE_RELU_BIAS : HIPBLASLT_EPILOGUE_RELU;
  else return LEV_LIBRARY_UNSUPPORTED;
  return 0;
}

int make_plan(hipblasLtHandle_t handle, Plan* p, int M, int N, int K, long lda, long ldr, long ldo, uint32_t epilogue, bool bias,
              bool residual, hipDataType out_type, size_t max_workspace) {
  LIB_CHECK(hipblasLtMatmulDescCreate(&p->desc, HIPBLAS_COMPUTE_32F, HIP_R_32F));
  const int32_t op_t = HIPBLAS_OP_T, op_n = HIPBLAS_OP_N;
  LIB_CHECK(hipblasLtMatmulDescSetAttribute(p->desc, HIPBLASLT_MATMUL_DESC_TRANSA, &op_t, sizeof(op_t)));
  LIB_CHECK(hipblasLtMatmulDescSetAttribute(p->desc, HIPBLASLT_MATMUL_DESC_TRANSB, &op_n, sizeof(op_n)));
  LIB_CHECK(hipblasLtMatmulDescSetAttribute(p->desc, HIPBLASLT_MATMUL_DESC_EPILOGUE, &epilogue, sizeof(epilogue)));
  if (bias) {
    const int32_t bias_type = HIP_R_32F;
    LIB_CHECK(hipblasLtMatmulDescSetAttribute(p->desc, HIPBLASLT_MATMUL_DESC_BIAS_DATA_TYPE, &bias_type, sizeof(bias_type)));
  }
  LIB_CHECK(hipblasLtMatrixLayoutCreate(&p->lw, HIP_R_16BF, K, N, K));
  LIB_CHECK(hipblasLtMatrixLayoutCreate(&p->la, HIP_R_16BF, K, M, lda));
  LIB_CHECK(hipblasLtMatrixLayoutCreate(&p->lc, out_type, N, M, residual ? ldr : ldo));
  LIB_CHECK(hipblasLtMatrixLayoutCreate(&p->ld, out_type, N, M, ldo));
  hipblasLtMatmulPreference_t pref = nullptr;
  LIB_CHECK(hipblasLtMatmulPreferenceCreate(&pref));
  const uint64_t ws = max_workspace;
  hipblasStatus_t s = hipblasLtMatmulPreferenceSetAttribute(pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &ws, sizeof(ws));
  hipblasLtMatmulHeuristicResult_t result[LEV_LIB_CANDIDATES];
  int found = 0;
  if (s == HIPBLAS_STATUS_SUCCESS)
    s = hipblasLtMatmulAlgoGetHeuristic(handle, p->desc, p->lw, p->la, p->lc, p->ld, pref, LEV_LIB_CANDIDATES, result, &found);
  hipblasLtMatmulPreferenceDestroy(pref);
  if (s != HIPBLAS_STATUS_SUCCESS || found < 1) return LEV_LIBRARY_UNSUPPORTED;  // p->ok stays false: remembered, not asked again
  for (int i = 0; i < found; ++i)
    if (result[i].state == HIPBLAS_STATUS_SUCCESS && result[i].workspaceSize <= max_workspace) p->candidates.push_back(result[i]);
  if (p->candidates.empty()) return LEV_LIBRARY_UNSUPPORTED;
  p->algo = p->candidates[0].algo;
  p->workspace = p->candidates[0].workspaceSize;
  p->ok = true;
  return 0;
}

// 0: the heuristic's first kernel is taken; 1 (default): the candidates of a shape are timed at its first call outside a
// stream capture and the fastest is kept; 2: the timings are printed as well.
int tune_level() {
  static const int level = [] {
    const char* e = getenv("LEVANTER_AMD_GEMM_TUNE");
    return e ? atoi(e) : 1;
  }();
  return level;
}

// A buffer larger than the caches (32 MB of L2, 256 MB behind them), one per device, kept for the life of the process:
// sweeping it between two timed runs leaves nothing of the operands in a cache. Ahead of them it holds bfloat16 numbers of either sign, 1/4 to 4, all bits
// of which vary: operands on which the kernels' sums are told apart.
#define LEV_LIB_FLUSH_BYTES ((size_t)512 << 20)
__global__ void __launch_bounds__(256) fill_kernel(uint4* to, uint32_t n) {
  auto mixed = [](uint32_t x) {
    x *= 0x9e3779b1u, x ^= x >> 15, x *= 0x85ebca77u, x ^= x >> 13;
    const uint32_t raise = x >> 1 & 0x01000100u;  // exponents 125 and 126, 127 and 128
    return (x & 0x80ff80ffu) + 0x3e803e80u + raise;
  };
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) to[i] = uint4{mixed(4 * i), mixed(4 * i + 1), mixed(4 * i + 2), mixed(4 * i + 3)};
}
bool fill(void* flush, hipStream_t stream) {
  fill_kernel<<<2048, 256, 0, stream>>>((uint4*)flush, (uint32_t)(LEV_LIB_FLUSH_BYTES / sizeof(uint4)));
  return hipGetLastError() == hipSuccess;
}
void* flush_buffer() {
  static std::map<int, void*> buffers;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
  auto it = buffers.find(dev);
  if (it != buffers.end()) return it->second;
  void* p = nullptr;
  if (hipMalloc(&p, LEV_LIB_FLUSH_BYTES) != hipSuccess) { (void)hipGetLastError(); p = nullptr; }
  buffers[dev] = p;
  return p;
}

// What tells two results' bits apart: their sum, each word times an odd number of its place.
template <class Word>
__global__ void __launch_bounds__(256) bits_kernel(const Word* __restrict__ y, int M, int N, long ldo, unsigned long long* sum) {
  unsigned long long t = 0;
  for (int m = blockIdx.x; m < M; m += gridDim.x)
    for (int n = threadIdx.x; n < N; n += 256) t += y[(size_t)m * ldo + n] * (((unsigned long long)m * N + n) * 0x9e3779b97f4a7c16ull + 1);
  for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
  if ((threadIdx.x & 63) == 0) atomicAdd(sum, t);
}

// Of n kernels with the given bits and times (negative: did not run) the one to keep, or -1. Kernels that deal a product's last tiles out over the CUs along K add its sums up in
// another order than those that do not, so that the choice decides the result's last bits, and these are not to hang on a stopwatch. So: an order of sums that a single
// kernel has counts only where no two share one, and one order is preferred to another only where its fastest kernel is ahead by more than LEV_LIB_AHEAD; otherwise
// the one that more kernels have, then the one of the heuristic's earlier kernel. Over 77 shapes of 257 .. 2,070 rows the orders that are left are 4.3 % apart or more
// where there is more than one (mostly all sixteen kernels share one), while the kernels were down to 0.2 %: 4096 x 16384 at 1,088 rows takes 176 us with two of the kernels, 183 and 188
// with one each, 198 with three that do not split; it was the one product of the 7B sizes whose bits went by the process. What this gives away: 50257 x 4096 from 900 rows on 4 - 6 %.
#define LEV_LIB_AHEAD 1.02f
extern "C" int lev_linear_library_keeps(const unsigned long long* bits, const float* us, int n) {
  struct Order { int kernels, first, best; };
  std::vector<Order> orders;
  for (int i = 0; i < n; ++i) {
    if (us[i] < 0.0f) continue;
    size_t at = 0;
    while (at < orders.size() && bits[orders[at].first] != bits[i]) ++at;
    if (at == orders.size()) orders.push_back({0, i, i});
    Order& o = orders[at];
    ++o.kernels;
    if (us[i] < us[o.best]) o.best = i;
  }
  bool shared = false;
  for (const Order& o : orders) shared |= o.kernels > 1;
  float fastest = -1.0f;
  for (const Order& o : orders)
    if ((!shared || o.kernels > 1) && (fastest < 0.0f || us[o.best] < fastest)) fastest = us[o.best];
  const Order* kept = nullptr;
  for (const Order& o : orders)
    if ((!shared || o.kernels > 1) && us[o.best] <= fastest * LEV_LIB_AHEAD && (!kept || o.kernels > kept->kernels)) kept = &o;
  return kept ? kept->best : -1;
}

int index_of(hipblasLtMatmulAlgo_t algo) { return hipblaslt_ext::getIndexFromAlgo(algo); }

// Rows of the call that a tile of the kernel has, from its name (_MT<outputs>x<rows>x<depth>_), or 0.
int tile_rows(hipblasLtHandle_t handle, hipblasLtMatmulAlgo_t algo) {
  const std::string name = hipblaslt_ext::getSolutionNameFromAlgo(handle, algo);
  const size_t at = name.find("_MT");
  int outputs, rows;
  return at != std::string::npos && sscanf(name.c_str() + at, "_MT%dx%dx", &outputs, &rows) == 2 && rows > 0 ? rows : 0;
}

// Runs of a plan's candidates on a call's operands, writing to a buffer of their own (a product into the residual stream adds to its output, so the real output
// cannot take repeated runs). Allocates and synchronises: used only outside a stream capture.
struct Trial {
  hipblasLtHandle_t handle;
  Plan* plan;
  const void *a, *w;
  const float *bias, *residual;
  void* workspace;
  int M, N, K, out_dtype;
  long lda, ldr, ldo;
  hipStream_t stream;
  void *scratch = nullptr, *flush = nullptr;
  unsigned long long* sums = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  unsigned long long bits[LEV_LIB_CANDIDATES];
  float us[LEV_LIB_CANDIDATES];  // microseconds; 0: ran, not timed; negative: did not run, or is not asked for
  bool loaded[LEV_LIB_CANDIDATES] = {};

  bool begin() {
    const size_t bytes = ((size_t)M * (size_t)ldo * (out_dtype == LEV_F32 ? 4 : 2) + 255) / 256 * 256;
    for (float& t : us) t = -1.0f;
    if (hipMalloc(&scratch, bytes + sizeof(bits)) != hipSuccess) { (void)hipGetLastError(); scratch = nullptr; return false; }
    sums = (unsigned long long*)((char*)scratch + bytes);
    flush = flush_buffer();  // null if it could not be had: the runs are then timed on a warm weight, and all on the call's operands
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) { (void)hipGetLastError(); return false; }
    return true;
  }
  ~Trial() {
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (!scratch) return;
    (void)hipStreamSynchronize(stream);
    (void)hipFree(scratch);
  }
  bool run(int i, const void* a_, const void* w_, const void* c_) {
    const float alpha = 1.0f, beta = residual ? 1.0f : 0.0f;
    loaded[i] = true;
    return hipblasLtMatmul(handle, plan->desc, &alpha, w_, plan->lw, a_, plan->la, &beta, residual ? c_ : scratch, plan->lc, scratch, plan->ld, &plan->candidates[i].algo, workspace,
                           plan->candidates[i].workspaceSize, stream) == HIPBLAS_STATUS_SUCCESS;
  }
  bool bias_at(const void* b) {
    return !bias || hipblasLtMatmulDescSetAttribute(plan->desc, HIPBLASLT_MATMUL_DESC_BIAS_POINTER, &b, sizeof(b)) == HIPBLAS_STATUS_SUCCESS;
  }
  // The bits of the given kernels' results, on the buffer's numbers where it has enough of them (the call's may be zeros, on which all are alike): a weight from another place
  // than the rows, which it may overlap. us becomes 0 where there are some.
  void tell_apart(const std::vector<int>& which) {
    const size_t w_at = ((size_t)1 << 20) + 4096;
    const bool ours = flush && fill(flush, stream) && ((size_t)M * lda) * 2 <= LEV_LIB_FLUSH_BYTES && w_at + (size_t)N * K * 2 <= LEV_LIB_FLUSH_BYTES &&
                      (size_t)M * ldr * 4 <= LEV_LIB_FLUSH_BYTES && bias_at(flush);
    bool all = hipMemsetAsync(sums, 0, sizeof(bits), stream) == hipSuccess;
    for (int i : which) {
      us[i] = all && (ours ? run(i, flush, (const char*)flush + w_at, flush) : run(i, a, w, residual)) ? 0.0f : -1.0f;
      if (us[i] < 0.0f) { (void)hipGetLastError(); continue; }
      if (out_dtype == LEV_F32) bits_kernel<uint32_t><<<1024, 256, 0, stream>>>((const uint32_t*)scratch, M, N, ldo, sums + i);
      else bits_kernel<uint16_t><<<1024, 256, 0, stream>>>((const uint16_t*)scratch, M, N, ldo, sums + i);
    }
    all = all && hipMemcpyAsync(bits, sums, sizeof(bits), hipMemcpyDeviceToHost, stream) == hipSuccess && hipStreamSynchronize(stream) == hipSuccess;
    all = bias_at(bias) && all;
    if (!all)
      for (int i : which) us[i] = -1.0f;
  }
  // Every timed run behind a sweep over a buffer larger than the caches: in a model's step a product's weight has not
  // been touched since the step before, and the kernel that is fastest on a weight that waits in the last-level cache
  // (what a plain loop over one weight measures) is often not the fastest on one that comes from memory. The fastest
  // of the runs counts; a kernel's first run loads it and does not.
  void time(int i) {
    bool ok = loaded[i] || run(i, a, w, residual);
    float ms = -1.0f;
    for (int r = 1; r <= LEV_LIB_TUNE_RUNS && ok; ++r) {
      float t = 0.0f;
      ok = (!flush || hipMemsetAsync(flush, r, LEV_LIB_FLUSH_BYTES, stream) == hipSuccess) && hipEventRecord(e0, stream) == hipSuccess && run(i, a, w, residual) &&
           hipEventRecord(e1, stream) == hipSuccess && hipEventSynchronize(e1) == hipSuccess && hipEventElapsedTime(&t, e0, e1) == hipSuccess;
      if (ok && (ms < 0.0f || t < ms)) ms = t;
    }
    us[i] = ok ? ms * 1000.0f : -1.0f;
    if (!ok) { (void)hipGetLastError(); (void)hipStreamSynchronize(stream); return; }
    if (tune_level() >= 2) fprintf(stderr, "linear (library) M=%d N=%d K=%d: candidate %d (kernel %d) %.1f us\n", M, N, K, i, index_of(plan->candidates[i].algo), us[i]);
  }
};

// Gives the plan the kernel to keep. The heuristic's order is a table look-up by size; on this chip its first kernel is often not the fastest one for the shape at hand.
//
// known: what another row count of the bucket keeps, or null. All kernels again would be most of a first call's time (12288 x 4096: 17 ms); the order of sums is that which two of
// the first three kernels of the known order have here too, and only the known kernel, where it has it, and the heuristic's first, where it has too, are timed (a kernel that won at 264 rows can lose at
// 320, where its tiles divide the rows differently). A kernel with as many rows of tiles as there deals them out as there: where that is so of all that count, nothing is run to tell them apart. All are
// tried again where the known kernel is not on offer or has another order (the heuristic's first was up to a third slower than the best at 304 and 320 rows of a 1600-wide layer, whose bucket was timed at 272).
Kept time_candidates(Trial& trial, const Kept* known) {
  Plan* p = trial.plan;
  p->timed = true;
  const std::vector<hipblasLtMatmulHeuristicResult_t>& candidates = p->candidates;
  const int n = (int)candidates.size();
  Kept kept;
  kept.rows = trial.M;
  if (n < 2) return kept;
  auto t_begin = std::chrono::steady_clock::now();
  auto keep = [&](int i) {
    p->algo = candidates[i].algo;
    p->workspace = candidates[i].workspaceSize;
    kept.index = index_of(p->algo);
    if (tune_level() >= 2)
      fprintf(stderr, "linear (library) M=%d N=%d K=%d: kept candidate %d after %.1f ms\n", trial.M, trial.N, trial.K, i,
              std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_begin).count());
    return kept;
  };
  auto place = [&](int index) {
    for (int i = 0; i < n; ++i)
      if (index_of(candidates[i].algo) == index) return i;
    return -1;
  };
  std::vector<int> members;  // of the known order
  if (known)
    for (size_t j = 0; j < known->order.size() && members.size() < 3; ++j)
      if (const int i = place(known->order[j]); i >= 0) members.push_back(i);
  const int theirs = known ? place(known->index) : -1;
  bool begun = false;
  if (theirs >= 0 && members.size() >= 2) {
    auto alike = [&](int i) {
      const int t = tile_rows(trial.handle, candidates[i].algo);
      return t > 0 && (trial.M + t - 1) / t == (known->rows + t - 1) / t;
    };
    bool all = alike(theirs), they = all, first = false;  // the known kernel has the order here, the heuristic's first has
    for (int i : members) all &= alike(i);
    if (all) {
      first = std::find(known->order.begin(), known->order.end(), index_of(candidates[0].algo)) != known->order.end() && alike(0);
    } else {
      they = false;
      if (!(begun = trial.begin())) return kept;
      std::vector<int> which = members;
      for (int i : {theirs, 0})
        if (std::find(which.begin(), which.end(), i) == which.end()) which.push_back(i);
      trial.tell_apart(which);
      auto same = [&](int i, int j) { return trial.us[i] >= 0.0f && trial.us[j] >= 0.0f && trial.bits[i] == trial.bits[j]; };
      for (size_t j = 0; j + 1 < members.size() && !they; ++j)
        for (size_t k = j + 1; k < members.size() && !they; ++k)
          if (same(members[j], members[k])) they = same(theirs, members[j]), first = same(0, members[j]);
    }
    if (they && (!first || theirs == 0)) return keep(theirs);
    if (they) {
      if (!begun && !(begun = trial.begin())) return kept;
      trial.time(theirs), trial.time(0);
      const float x = trial.us[theirs], y = trial.us[0];
      if (x >= 0.0f || y >= 0.0f) return keep(y < 0.0f || (x >= 0.0f && x <= y) ? theirs : 0);
      return kept;
    }
  }
  if (!begun && !(begun = trial.begin())) return kept;
  std::vector<int> which;
  for (int i = 0; i < n; ++i) which.push_back(i);
  trial.tell_apart(which);
  bool shared = false, alone[LEV_LIB_CANDIDATES];
  for (int i = 0; i < n; ++i) {
    alone[i] = true;
    for (int j = 0; j < n; ++j) alone[i] &= !(i != j && trial.us[i] >= 0.0f && trial.us[j] >= 0.0f && trial.bits[i] == trial.bits[j]);
    shared |= !alone[i];
  }
  bool ran[LEV_LIB_CANDIDATES];
  for (int i = 0; i < n; ++i) {
    ran[i] = trial.us[i] >= 0.0f;
    if (ran[i] && shared && alone[i]) trial.us[i] = -1.0f;  // not to be kept
    else if (ran[i]) trial.time(i);
  }
  const int best = lev_linear_library_keeps(trial.bits, trial.us, n);
  if (best < 0) return kept;
  for (int i = 0; i < n; ++i)
    if (ran[i] && trial.bits[i] == trial.bits[best]) kept.order.push_back(index_of(candidates[i].algo));
  return keep(best);
}

// The kernel that timing chose for another row count of the plan's bucket, if the heuristic offers it for this row count
// too. (Asking the library for a kernel by its index instead makes it load its whole catalogue: a second at its first use.)
const hipblasLtMatmulHeuristicResult_t* candidate_of_index(const Plan* p, int index) {
  for (const hipblasLtMatmulHeuristicResult_t& cand : p->candidates) {
    hipblasLtMatmulAlgo_t algo = cand.algo;
    if (hipblaslt_ext::getIndexFromAlgo(algo) == index) return &cand;
  }
  return nullptr;
}

}  // namespace

// Bytes of workspace the caller must bring (one size for every shape: the heuristic is asked for kernels within it).
extern "C" long lev_linear_library_workspace() { return 64L << 20; }

// Returns 0 (done), LEV_LIBRARY_UNSUPPORTED (nothing was launched: run the hand-written kernel) or -1 with a message.
extern "C" int lev_linear_library(const void* a, long lda, const void* w, const float* bias, const float* residual, long ldr,
                                  void* out, long ldo, void* workspace, long workspace_bytes, int M, int N, int K, int act,
                                  int out_dtype, hipStream_t stream) {
  LEV_REQUIRE(M > 0 && N > 0 && K > 0, "linear (library): bad sizes M=%d N=%d K=%d", M, N, K);
  LEV_REQUIRE(lda >= K && ldo >= N, "linear (library): row strides lda=%ld ldo=%ld are smaller than K=%d / N=%d", lda, ldo, K, N);
  LEV_REQUIRE(!residual || (ldr >= N && out_dtype == LEV_F32), "linear (library): a residual needs a float32 output and a row stride >= N");
  LEV_REQUIRE(out_dtype == LEV_F32 || out_dtype == LEV_BF16, "linear (library): unknown output dtype %d", out_dtype);
  uint32_t epilogue;
  if (epilogue_of(act, bias != nullptr, &epilogue)) return LEV_LIBRARY_UNSUPPORTED;
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= LEV_LIB_MAX_DEVICES) return lev_fail("linear (library): no current device");
  // One lock for the look-up, the bias pointer (the descriptor is shared by every call of this shape) and the launch.
  std::lock_guard<std::mutex> lock(g_mutex);
  if (!g_handle[dev]) LIB_CHECK(hipblasLtCreate(&g_handle[dev]));
  hipblasLtHandle_t handle = g_handle[dev];
  const PlanKey key(dev, M, N, K, lda, residual ? ldr : 0, ldo, (int)epilogue, out_dtype, residual ? 1 : 0);
  auto it = g_plans.find(key);
  if (it == g_plans.end()) {
    Plan p;
    const int rc = make_plan(handle, &p, M, N, K, lda, ldr, ldo, epilogue, bias != nullptr, residual != nullptr,
                             out_dtype == LEV_F32 ? HIP_R_32F : HIP_R_16BF, (size_t)workspace_bytes);
    if (rc < 0) return rc;
    it = g_plans.emplace(key, p).first;
  }
  Plan& plan = it->second;
  if (!plan.ok) return LEV_LIBRARY_UNSUPPORTED;
  if (bias) {
    const void* bp = bias;
    LIB_CHECK(hipblasLtMatmulDescSetAttribute(plan.desc, HIPBLASLT_MATMUL_DESC_BIAS_POINTER, &bp, sizeof(bp)));
  }
  if (!plan.timed && M >= LEV_LIB_TUNE_MIN_ROWS && tune_level() >= 1) {
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capturing) != hipSuccess) { (void)hipGetLastError(); capturing = hipStreamCaptureStatusActive; }
    const bool may_time = capturing == hipStreamCaptureStatusNone;
    const PlanKey bucket(dev, rows_bucket(M), N, K, lda, residual ? ldr : 0, ldo, (int)epilogue, out_dtype, residual ? 1 : 0);
    auto known = g_kept.find(bucket);
    if (may_time) {
      Trial trial{handle, &plan, a, w, bias, residual, workspace, M, N, K, out_dtype, lda, ldr, ldo, stream};
      Kept kept = time_candidates(trial, known == g_kept.end() ? nullptr : &known->second);
      if (known == g_kept.end()) g_kept[bucket] = kept;
    } else {
      plan.timed = true;  // recorded into a graph with the heuristic's first kernel, or the one its bucket keeps: eager calls of this shape keep it
                          // too, so that a replay and an eager run of the same product give the same bits
      if (known != g_kept.end() && known->second.index >= 0)
        if (const hipblasLtMatmulHeuristicResult_t* theirs = candidate_of_index(&plan, known->second.index)) {
          plan.algo = theirs->algo;
          plan.workspace = theirs->workspaceSize;
        }
    }
  }
  if (plan.workspace > 0 && !workspace)
    return lev_fail("linear (library): the chosen kernel needs %zu bytes of workspace, none was brought", plan.workspace);
  const float alpha = 1.0f, beta = residual ? 1.0f : 0.0f;
  LIB_CHECK(hipblasLtMatmul(handle, plan.desc, &alpha, w, plan.lw, a, plan.la, &beta, residual ? (const void*)residual : (const void*)out,
                            plan.lc, out, plan.ld, &plan.algo, workspace, plan.workspace, stream));
  return 0;
}
