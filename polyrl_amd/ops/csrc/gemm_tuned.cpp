// Per-shape hipBLASLt algo search for the trainer's hot GEMMs (host code).
//
// Why: hipBLASLt's default heuristic picks algorithms that are 20 to 45% off for the
// trainer's shapes (nt of some 7000 rows 0.88 to 1.27 PFLOP/s where the best runs at 1.6),
// and tables of algorithms from one machine do not hold on another.  On the first call
// for a (layout, M, N, K) key a list of candidates is asked for, each is timed on the
// live stream, and the winner is kept for the process's life.  No files, bounded cost
// (at most 48 algorithms, 4 runs each, once a shape).
//
// Reference capability: the update-loop GEMM throughput the reference gets
// from cuBLAS/flash-attn inside torch (stream_dp_actor.py:153-224).
//
// Layout math (row-major tensors on a column-major BLAS):
//   fwd  (nt): Y[M,N] = X[M,K] @ W[N,K]^T  ->  C(N,M) = op_T(W) op_N(X)
//   dgrad(nn): dX[M,K] = dY[M,N] @ W[N,K]  ->  C(K,M) = op_N(W) op_N(dY)
//   wgrad(tn): dW[N,K] = dY[M,N]^T @ X[M,K]->  C(K,N) = op_N(X) op_T(dY)
// Most gradients of many rows are the kernels' in linear_backward.hip, and the forward
// product of linear_prompt.hip is one more candidate: it is timed against the best
// algorithm with operands that the caches do not hold, as a layer finds its weight.
// (Repeated on one weight the two are often within 3% where memory parts them: 8192 ->
// 8192 of 513 rows 73 and 73 us repeated, 103 and 85 from memory; 18944 -> 3584 of 1536
// 181 and 180, 231 and 205; 4096 -> 14336 of 4096 350 and 349, 373 and 348.  Where tiles of
// 256 rows are not whole it takes 0.86 to 0.98 of the algorithm's time: 7168 rows, 4096 ->
// 14336, 14336 -> 4096, 4096 -> 4096 559, 542, 158 us for 575, 576, 164.)
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <hipblaslt/hipblaslt.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#define HIPBLASLT_CHECK(expr)                                             \
  do {                                                                    \
    hipblasStatus_t s_ = (expr);                                          \
    TORCH_CHECK(s_ == HIPBLAS_STATUS_SUCCESS, "hipblaslt error ", (int)s_, \
                " at " #expr);                                            \
  } while (0)

// linear_backward.hip
bool linear_wgrad_takes(const torch::Tensor& dy, const torch::Tensor& x);
bool linear_dgrad_takes(const torch::Tensor& dy, const torch::Tensor& w);
torch::Tensor linear_wgrad(torch::Tensor dy, torch::Tensor x);
torch::Tensor linear_dgrad(torch::Tensor dy, torch::Tensor w);
// linear_prompt.hip
bool linear_rows_fits(const torch::Tensor& x, const torch::Tensor& w);
void linear_rows_into(torch::Tensor& out, const torch::Tensor& x,
                      const torch::Tensor& w);

namespace {

constexpr size_t kWorkspaceBytes = 128ull << 20;
constexpr int kMaxAlgos = 48;
constexpr int kTimedIters = 3;
constexpr int64_t kKernelRows = 513;   // fewer leave the kernel's tiles empty
constexpr int64_t kFlushBytes = 512ll << 20;   // twice what the last cache holds

struct Pick {
  hipblasLtMatmulAlgo_t algo;
  bool kernel;                         // linear_prompt.hip's is the faster one
};

struct LtState {
  hipblasLtHandle_t handle = nullptr;
  std::mutex mu;
  // key: (mode, M, N, K) -> winning algo
  std::map<std::tuple<int, int64_t, int64_t, int64_t>, Pick> cache;
};

// (what was found can be asked for where no GPU is)
LtState& lt_state() {
  static LtState s;
  return s;
}

LtState& lt() {
  auto& s = lt_state();
  static std::once_flag once;
  std::call_once(once, [&] { HIPBLASLT_CHECK(hipblasLtCreate(&s.handle)); });
  return s;
}

// Workspace is per-THREAD: each thread in this stack owns its stream
// (trainer main, engine pump, uvicorn handlers), and a shared workspace
// would be written concurrently by matmuls running on different streams.
void* tl_workspace() {
  static thread_local void* ws = nullptr;
  if (ws == nullptr)
    TORCH_CHECK(hipMalloc(&ws, kWorkspaceBytes) == hipSuccess,
                "hipblaslt workspace alloc failed");
  return ws;
}

struct Plan {
  hipblasLtMatmulDesc_t op = nullptr;
  hipblasLtMatrixLayout_t la = nullptr, lb = nullptr, lc = nullptr;
  ~Plan() {
    if (op) hipblasLtMatmulDescDestroy(op);
    if (la) hipblasLtMatrixLayoutDestroy(la);
    if (lb) hipblasLtMatrixLayoutDestroy(lb);
    if (lc) hipblasLtMatrixLayoutDestroy(lc);
  }
};

// column-major problem: C(m,n) = opA(A) * opB(B)
void build_plan(Plan& p, hipblasOperation_t opA, hipblasOperation_t opB,
                int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb,
                int64_t ldc) {
  HIPBLASLT_CHECK(hipblasLtMatmulDescCreate(&p.op, HIPBLAS_COMPUTE_32F,
                                            HIP_R_32F));
  HIPBLASLT_CHECK(hipblasLtMatmulDescSetAttribute(
      p.op, HIPBLASLT_MATMUL_DESC_TRANSA, &opA, sizeof(opA)));
  HIPBLASLT_CHECK(hipblasLtMatmulDescSetAttribute(
      p.op, HIPBLASLT_MATMUL_DESC_TRANSB, &opB, sizeof(opB)));
  const int64_t ra = (opA == HIPBLAS_OP_N) ? m : k;
  const int64_t ca = (opA == HIPBLAS_OP_N) ? k : m;
  const int64_t rb = (opB == HIPBLAS_OP_N) ? k : n;
  const int64_t cb = (opB == HIPBLAS_OP_N) ? n : k;
  HIPBLASLT_CHECK(hipblasLtMatrixLayoutCreate(&p.la, HIP_R_16BF, ra, ca, lda));
  HIPBLASLT_CHECK(hipblasLtMatrixLayoutCreate(&p.lb, HIP_R_16BF, rb, cb, ldb));
  HIPBLASLT_CHECK(hipblasLtMatrixLayoutCreate(&p.lc, HIP_R_16BF, m, n, ldc));
}

// Whether ``kernel`` is faster than ``library`` with its weight in memory, and x where the
// layer before it left it: the best of some runs of each, in turn.  ``kernel`` runs last.
// (No where there is no memory to pass through the caches.)
template <typename Kernel, typename Library>
bool faster_from_memory(const torch::Tensor& x, Kernel kernel, Library library,
                        hipEvent_t ev0, hipEvent_t ev1, hipStream_t stream) {
  torch::Tensor flush, copy;
  try {
    flush = torch::empty({kFlushBytes}, x.options().dtype(torch::kUInt8));
    copy = torch::empty_like(x);
  } catch (const c10::OutOfMemoryError&) {
    return false;
  }
  auto time = [&](auto& run) {
    flush.fill_(1);
    copy.copy_(x);
    hipEventRecord(ev0, stream);
    run();
    hipEventRecord(ev1, stream);
    hipEventSynchronize(ev1);
    float ms = 1e30f;
    hipEventElapsedTime(&ms, ev0, ev1);
    return ms;
  };
  float of_kernel = 1e30f, of_library = 1e30f;
  library(), kernel();                 // (code and tables are loaded once)
  for (int i = 0; i < kTimedIters; ++i) {
    of_library = std::min(of_library, time(library));
    of_kernel = std::min(of_kernel, time(kernel));
  }
  return of_kernel < of_library;
}

// mode: 0 = fwd nt, 1 = dgrad nn, 2 = wgrad tn
void tuned_mm(int mode, const torch::Tensor& A_row, const torch::Tensor& B_row,
              torch::Tensor& C_row, int64_t M, int64_t N, int64_t K) {
  auto& s = lt();
  void* workspace = tl_workspace();
  auto stream = at::hip::getCurrentHIPStream();

  hipblasOperation_t opA, opB;
  int64_t m, n, k, lda, ldb, ldc;
  const void *Aptr, *Bptr;
  void* Cptr = C_row.data_ptr();
  if (mode == 0) {           // C(N,M) = W^T(cm K,N) X(cm K,M)
    opA = HIPBLAS_OP_T; opB = HIPBLAS_OP_N;
    m = N; n = M; k = K; lda = K; ldb = K; ldc = N;
    Aptr = B_row.data_ptr();  // W
    Bptr = A_row.data_ptr();  // X
  } else if (mode == 1) {    // C(K,M) = W(cm K,N) dY(cm N,M)
    opA = HIPBLAS_OP_N; opB = HIPBLAS_OP_N;
    m = K; n = M; k = N; lda = K; ldb = N; ldc = K;
    Aptr = B_row.data_ptr();  // W
    Bptr = A_row.data_ptr();  // dY
  } else {                   // C(K,N) = X(cm K,M) dY^T(cm N,M)
    opA = HIPBLAS_OP_N; opB = HIPBLAS_OP_T;
    m = K; n = N; k = M; lda = K; ldb = N; ldc = K;
    Aptr = B_row.data_ptr();  // X
    Bptr = A_row.data_ptr();  // dY
  }

  // (an address of another alignment than the searched one's has the algorithm)
  const bool kernel_fits =
      mode == 0 && M >= kKernelRows && linear_rows_fits(A_row, B_row);
  Pick pick;
  bool have_algo = false;
  {
    std::lock_guard<std::mutex> g(s.mu);
    auto it = s.cache.find({mode, M, N, K});
    if (it != s.cache.end()) {
      pick = it->second;
      have_algo = true;
    }
  }
  if (have_algo && pick.kernel && kernel_fits) {
    linear_rows_into(C_row, A_row, B_row);
    return;
  }

  Plan p;
  build_plan(p, opA, opB, m, n, k, lda, ldb, ldc);
  const float alpha = 1.f, beta = 0.f;

  if (!have_algo) {
    hipblasLtMatmulPreference_t pref;
    HIPBLASLT_CHECK(hipblasLtMatmulPreferenceCreate(&pref));
    size_t ws = kWorkspaceBytes;
    HIPBLASLT_CHECK(hipblasLtMatmulPreferenceSetAttribute(
        pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &ws, sizeof(ws)));
    std::vector<hipblasLtMatmulHeuristicResult_t> results(kMaxAlgos);
    int found = 0;
    HIPBLASLT_CHECK(hipblasLtMatmulAlgoGetHeuristic(
        s.handle, p.op, p.la, p.lb, p.lc, p.lc, pref, kMaxAlgos,
        results.data(), &found));
    hipblasLtMatmulPreferenceDestroy(pref);
    TORCH_CHECK(found > 0, "hipblaslt: no algo for shape mode=", mode,
                " M=", M, " N=", N, " K=", K);

    hipEvent_t ev0, ev1;
    hipEventCreate(&ev0);
    hipEventCreate(&ev1);
    float best_ms = 1e30f;
    int best = 0;
    for (int i = 0; i < found; ++i) {
      // warmup (also validates the algo actually runs)
      hipblasStatus_t st = hipblasLtMatmul(
          s.handle, p.op, &alpha, Aptr, p.la, Bptr, p.lb, &beta, Cptr, p.lc,
          Cptr, p.lc, &results[i].algo, workspace, kWorkspaceBytes, stream);
      if (st != HIPBLAS_STATUS_SUCCESS) continue;
      hipEventRecord(ev0, stream);
      for (int it2 = 0; it2 < kTimedIters; ++it2)
        hipblasLtMatmul(s.handle, p.op, &alpha, Aptr, p.la, Bptr, p.lb,
                        &beta, Cptr, p.lc, Cptr, p.lc, &results[i].algo,
                        workspace, kWorkspaceBytes, stream);
      hipEventRecord(ev1, stream);
      hipEventSynchronize(ev1);
      float ms = 1e30f;
      hipEventElapsedTime(&ms, ev0, ev1);
      if (ms < best_ms) {
        best_ms = ms;
        best = i;
      }
    }
    pick.kernel =
        kernel_fits && best_ms < 1e29f &&
        faster_from_memory(
            A_row, [&] { linear_rows_into(C_row, A_row, B_row); },
            [&] {
              hipblasLtMatmul(s.handle, p.op, &alpha, Aptr, p.la, Bptr, p.lb, &beta,
                              Cptr, p.lc, Cptr, p.lc, &results[best].algo, workspace,
                              kWorkspaceBytes, stream);
            },
            ev0, ev1, stream);
    hipEventDestroy(ev0);
    hipEventDestroy(ev1);
    TORCH_CHECK(best_ms < 1e29f, "hipblaslt: every candidate failed, mode=",
                mode, " M=", M, " N=", N, " K=", K);
    pick.algo = results[best].algo;
    {
      std::lock_guard<std::mutex> g(s.mu);
      s.cache[{mode, M, N, K}] = pick;
    }
    if (pick.kernel) return;           // (its product is the one there)
  }

  HIPBLASLT_CHECK(hipblasLtMatmul(
      s.handle, p.op, &alpha, Aptr, p.la, Bptr, p.lb, &beta, Cptr, p.lc,
      Cptr, p.lc, &pick.algo, workspace, kWorkspaceBytes, stream));
}

void check2d(const torch::Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda() && t.dim() == 2 && t.is_contiguous() &&
                  t.dtype() == torch::kBFloat16,
              name, " must be contiguous 2-D bf16 on GPU");
}

}  // namespace

// What the search found for Y = X W^T: 1 the kernel, 0 an algorithm, -1 not searched yet
long tuned_linear_pick(long M, long N, long K) {
  auto& s = lt_state();
  std::lock_guard<std::mutex> g(s.mu);
  auto it = s.cache.find({0, M, N, K});
  return it == s.cache.end() ? -1 : it->second.kernel;
}

// Y[M,N] = X[M,K] @ W[N,K]^T
torch::Tensor tuned_linear_fwd(torch::Tensor x, torch::Tensor w) {
  check2d(x, "x");
  check2d(w, "w");
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(w.size(1) == K, "shape mismatch");
  auto y = torch::empty({M, N}, x.options());
  tuned_mm(0, x, w, y, M, N, K);
  return y;
}

// dX[M,K] = dY[M,N] @ W[N,K]
torch::Tensor tuned_linear_dgrad(torch::Tensor dy, torch::Tensor w) {
  check2d(dy, "dy");
  check2d(w, "w");
  const int64_t M = dy.size(0), N = dy.size(1), K = w.size(1);
  TORCH_CHECK(w.size(0) == N, "shape mismatch");
  if (linear_dgrad_takes(dy, w)) return linear_dgrad(dy, w);
  auto dx = torch::empty({M, K}, dy.options());
  tuned_mm(1, dy, w, dx, M, N, K);
  return dx;
}

// dW[N,K] = dY[M,N]^T @ X[M,K]
torch::Tensor tuned_linear_wgrad(torch::Tensor dy, torch::Tensor x) {
  check2d(dy, "dy");
  check2d(x, "x");
  const int64_t M = dy.size(0), N = dy.size(1), K = x.size(1);
  TORCH_CHECK(x.size(0) == M, "shape mismatch");
  if (linear_wgrad_takes(dy, x)) return linear_wgrad(dy, x);
  auto dw = torch::empty({N, K}, dy.options());
  tuned_mm(2, dy, x, dw, M, N, K);
  return dw;
}
