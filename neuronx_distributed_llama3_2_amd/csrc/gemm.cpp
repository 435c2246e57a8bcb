// Autotuned hipBLASLt GEMM for the training / inference linear layers (gfx950).
//
// D = alpha * A @ B + beta * C for 2-D row-major-or-column-major views A [M,K], B [K,N] (bf16) and
// a row-major D [M,N] (bf16 or fp32, beta = 1 accumulates in place — the fp32 `main_grad`
// weight-gradient accumulation of the backward pass).
//
// Why not torch.matmul: PyTorch takes hipBLASLt's FIRST heuristic solution, and for the
// mixed-precision accumulate (bf16 x bf16 -> += fp32) that solution is a 256x256x32 macro tile
// running ~1.1 PF/s on MI355X.  Here every new problem (shape, strides, dtypes, beta) is timed over
// the top-N heuristic candidates with HIP events the first time it is seen (never while a stream is
// being captured into a hipGraph); the winner is cached in memory and, as its rank in the
// heuristic list, optionally in a text file (NXD_GEMM_TUNE_FILE) so later runs skip the timing
// (the algo is re-resolved by one heuristic query per shape — raw algo blobs are not valid across
// processes).  Tuning an accumulating GEMM writes into a scratch D so the real accumulator is only
// touched once.

#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <hip/hip_runtime.h>
#include <hipblaslt/hipblaslt-ext.hpp>
#include <hipblaslt/hipblaslt.h>
#include <torch/extension.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <map>
#include <mutex>
#include <sstream>
#include <string>
#include <unordered_map>
#include <unordered_set>
#include <vector>

namespace nxd {
int act_gemm_launch(int, const void*, const void*, void*, int64_t, int64_t, int64_t, hipStream_t);
}

namespace nxd_gemm {

#define LT_CHECK(x)                                                                          \
  do {                                                                                       \
    hipblasStatus_t _s = (x);                                                                \
    TORCH_CHECK(_s == HIPBLAS_STATUS_SUCCESS, "hipBLASLt error ", (int)_s, " at " #x);        \
  } while (0)

struct Problem {
  int opA, opB;             // hipBLASLt (column-major) ops
  int64_t m, n, k;          // column-major problem
  int64_t rowsA, colsA, lda, rowsB, colsB, ldb, ldc, ldd;
  int ta, tc;               // input / output hipDataType
  int beta_nonzero;
  bool no_sk = false;
  bool in_place = false;    // C and D are the same memory (the fp32 main_grad accumulation)
  int align = 256;          // smallest power-of-two alignment (<= 256 B) of the A / B / C / D pointers
  std::string key() const {
    std::ostringstream s;
    s << opA << ' ' << opB << ' ' << m << ' ' << n << ' ' << k << ' ' << lda << ' ' << ldb << ' ' << ldc << ' ' << ldd
      << ' ' << ta << ' ' << tc << ' ' << beta_nonzero << (no_sk ? " nosk" : "");
    // a solution validated at one pointer alignment / aliasing is not assumed valid at another
    // (the exhaustive search's choices are checked on exactly this call's layout)
    if (align < 256) s << " al" << align;
    if (beta_nonzero && in_place) s << " ip";
    return s.str();
  }
};

struct Choice {
  hipblasLtMatmulAlgo_t algo;
  size_t ws = 0;
  float ms = 0.f;
  int pos = 0;          // rank of the winner in the heuristic list (what the tune file stores)
  int index = -1;       // exhaustive mode: the library's global solution index ("i<index>" in files)
  bool resolved = false;  // algo blob valid in this process
};

class Tuner {
 public:
  static Tuner& get() {
    static Tuner t;
    return t;
  }

  hipblasLtHandle_t handle() {
    int dev = 0;
    (void)hipGetDevice(&dev);
    std::lock_guard<std::mutex> g(mu_);
    if ((int)handles_.size() <= dev) handles_.resize(dev + 1, nullptr);
    if (!handles_[dev]) LT_CHECK(hipblasLtCreate(&handles_[dev]));
    return handles_[dev];
  }

  // one workspace per (device, stream): GEMMs on concurrent streams (the two sequence-parallel
  // halves of parallel_layers/stream_split.py) must not share split-K / stream-K partials
  void* workspace(size_t bytes, hipStream_t stream) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    std::lock_guard<std::mutex> g(mu_);
    at::Tensor& w = ws_[std::make_pair(dev, (uintptr_t)stream)];
    if (w.numel() < (int64_t)bytes) {
      w = at::empty({(int64_t)bytes}, at::TensorOptions().dtype(at::kByte).device(at::kCUDA, dev));
    }
    return w.data_ptr();
  }

  size_t max_ws() const { return ws_limit_; }
  int retime() const { return retime_; }
  int candidates() const { return candidates_; }
  int mode() const { return mode_; }

  bool lookup(const std::string& key, Choice* out) {
    std::lock_guard<std::mutex> g(mu_);
    load_file_locked();
    auto it = cache_.find(key);
    if (it == cache_.end()) return false;
    *out = it->second;
    return true;
  }

  void store(const std::string& key, const Choice& c, bool persist) {
    std::lock_guard<std::mutex> g(mu_);
    cache_[key] = c;
    if (persist && !file_.empty()) {
      std::ofstream f(file_, std::ios::app);
      if (f) {
        if (c.index >= 0)
          f << key << " | i" << c.index << ' ' << c.ms << '\n';
        else
          f << key << " | " << c.pos << ' ' << c.ms << '\n';
      }
    }
  }

  std::vector<std::pair<std::string, float>> entries() {
    std::lock_guard<std::mutex> g(mu_);
    std::vector<std::pair<std::string, float>> v;
    for (auto& kv : cache_) v.emplace_back(kv.first, kv.second.ms);
    return v;
  }

 private:
  Tuner() {
    const char* m = std::getenv("NXD_GEMM_TUNE");
    mode_ = m ? std::atoi(m) : 1;  // 0: first heuristic, 1: time the top-N heuristics, 2: time every solution
    const char* t = std::getenv("NXD_GEMM_TABLE");  // read-only shipped table (tools/tune_gemm.py)
    if (t) table_ = t;
    const char* lk = std::getenv("NXD_GEMM_LOG_KEYS");
    if (lk) log_ = lk;
    const char* mx = std::getenv("NXD_GEMM_TUNE_MAX_ALGOS");
    max_algos_ = mx ? std::max(1, std::atoi(mx)) : 4096;
    const char* c = std::getenv("NXD_GEMM_TUNE_CANDIDATES");
    candidates_ = c ? std::max(1, std::atoi(c)) : 24;
    const char* f = std::getenv("NXD_GEMM_TUNE_FILE");
    if (f) file_ = f;
    const char* rt = std::getenv("NXD_GEMM_RETIME");
    retime_ = rt ? std::max(0, std::atoi(rt)) : 0;
    const char* w = std::getenv("NXD_GEMM_WORKSPACE_MB");
    ws_limit_ = (size_t)(w ? std::atoi(w) : 128) << 20;
  }

  void load_file_locked() {
    if (loaded_) return;
    loaded_ = true;
    for (const std::string* path : {&table_, &file_}) {  // later entries (the tune file) win
      if (path->empty()) continue;
      std::ifstream f(*path);
      std::string line;
      while (std::getline(f, line)) {
        auto bar = line.find('|');
        if (bar == std::string::npos) continue;
        std::string key = line.substr(0, bar);
        while (!key.empty() && key.back() == ' ') key.pop_back();
        std::istringstream s(line.substr(bar + 1));
        std::string tok;
        Choice c;
        if (!(s >> tok >> c.ms)) continue;
        if (!tok.empty() && tok[0] == 'i')
          c.index = std::atoi(tok.c_str() + 1);
        else
          c.pos = std::atoi(tok.c_str());
        cache_[key] = c;  // resolved lazily (by solution index, or heuristic query + pick pos)
      }
    }
  }

 public:
  int max_algos() const { return max_algos_; }

  // NXD_GEMM_LOG_KEYS=<file>: append every problem key this process meets (once) — the input of
  // tools/tune_gemm.py, which tunes each key offline and writes the shipped table
  void log_key(const std::string& key) {
    std::lock_guard<std::mutex> g(mu_);
    if (log_.empty() || !logged_.insert(key).second) return;
    std::ofstream f(log_, std::ios::app);
    if (f) f << key << '\n';
  }

 private:

  std::mutex mu_;
  std::vector<hipblasLtHandle_t> handles_;
  std::map<std::pair<int, uintptr_t>, at::Tensor> ws_;
  std::unordered_map<std::string, Choice> cache_;
  std::string file_, table_, log_;
  std::unordered_set<std::string> logged_;
  int max_algos_ = 4096;
  bool loaded_ = false;
  int mode_ = 1, candidates_ = 24, retime_ = 0;
  size_t ws_limit_ = 128u << 20;
};

// Overlap-safe selection (NXD_GEMM_NO_STREAMK / gemm_set_no_streamk): skip hipBLASLt's stream-K
// solutions ("_SK<n>" in the kernel name).  A stream-K GEMM runs one persistent workgroup per CU
// whose partial tiles are fixed up by the others; when a concurrent kernel (an RCCL channel, one
// workgroup) holds a CU, the fix-ups wait for the displaced workgroup and the GEMM takes ~1.8x as
// long (TP=8 gate_up / o_proj shapes with 4 side workgroups, profiles/r3_cu_interference.jsonl),
// where a data-parallel tile kernel only loses its tail.  Multi-rank training (collectives
// overlapping GEMMs) turns it on; -1 = not set (env, else off).
static int g_no_streamk = -1;
static bool no_streamk() {
  if (g_no_streamk < 0) {
    const char* e = std::getenv("NXD_GEMM_NO_STREAMK");
    g_no_streamk = (e && std::atoi(e) > 0) ? 1 : 0;
  }
  return g_no_streamk == 1;
}
static bool is_streamk(hipblasLtHandle_t h, hipblasLtMatmulAlgo_t algo) {
  const std::string n = hipblaslt_ext::getKernelNameFromAlgo(h, algo);
  for (size_t i = n.find("_SK"); i != std::string::npos; i = n.find("_SK", i + 1))
    if (i + 3 < n.size() && n[i + 3] >= '1' && n[i + 3] <= '9') return true;
  return false;
}

static hipDataType dt(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return HIP_R_16BF;
    case at::kHalf: return HIP_R_16F;
    case at::kFloat: return HIP_R_32F;
    default: TORCH_CHECK(false, "gemm: unsupported dtype ", t.scalar_type());
  }
  return HIP_R_32F;
}

struct Descs {
  hipblasLtMatmulDesc_t op = nullptr;
  hipblasLtMatrixLayout_t A = nullptr, B = nullptr, C = nullptr, D = nullptr;
  ~Descs() {
    if (A) hipblasLtMatrixLayoutDestroy(A);
    if (B) hipblasLtMatrixLayoutDestroy(B);
    if (C) hipblasLtMatrixLayoutDestroy(C);
    if (D) hipblasLtMatrixLayoutDestroy(D);
    if (op) hipblasLtMatmulDescDestroy(op);
  }
};

static void make_descs(const Problem& p, Descs& d) {
  LT_CHECK(hipblasLtMatmulDescCreate(&d.op, HIPBLAS_COMPUTE_32F, HIP_R_32F));
  hipblasOperation_t oa = (hipblasOperation_t)p.opA, ob = (hipblasOperation_t)p.opB;
  LT_CHECK(hipblasLtMatmulDescSetAttribute(d.op, HIPBLASLT_MATMUL_DESC_TRANSA, &oa, sizeof(oa)));
  LT_CHECK(hipblasLtMatmulDescSetAttribute(d.op, HIPBLASLT_MATMUL_DESC_TRANSB, &ob, sizeof(ob)));
  LT_CHECK(hipblasLtMatrixLayoutCreate(&d.A, (hipDataType)p.ta, p.rowsA, p.colsA, p.lda));
  LT_CHECK(hipblasLtMatrixLayoutCreate(&d.B, (hipDataType)p.ta, p.rowsB, p.colsB, p.ldb));
  LT_CHECK(hipblasLtMatrixLayoutCreate(&d.C, (hipDataType)p.tc, p.m, p.n, p.ldc));
  LT_CHECK(hipblasLtMatrixLayoutCreate(&d.D, (hipDataType)p.tc, p.m, p.n, p.ldd));
}

// Column-major view (rows, cols, ld, op) of the transpose of a row-major-or-column-major 2-D
// tensor X [R, S]: returns a layout for X^T (S x R).
static void transposed_view(const at::Tensor& x, int64_t* rows, int64_t* cols, int64_t* ld, int* op) {
  const int64_t R = x.size(0), S = x.size(1);
  const int64_t sR = x.stride(0), sS = x.stride(1);
  if (sS == 1 && (sR >= std::max<int64_t>(S, 1) || R == 1)) {  // row-major X == column-major X^T
    *rows = S; *cols = R; *ld = std::max<int64_t>(sR, S); *op = HIPBLAS_OP_N;
  } else if (sR == 1 && (sS >= std::max<int64_t>(R, 1) || S == 1)) {  // column-major X: X^T = op T of (R x S)
    *rows = R; *cols = S; *ld = std::max<int64_t>(sS, R); *op = HIPBLAS_OP_T;
  } else {
    TORCH_CHECK(false, "gemm: operand must have a unit stride in one dimension");
  }
}

static int ptr_align(const void* p) {
  const uintptr_t v = (uintptr_t)p;
  int a = 256;
  while (a > 1 && (v % a)) a >>= 1;
  return a;
}

// A scratch tensor shaped / strided like `like` whose data pointer has the same alignment mod
// 256 B: exhaustive candidates are validated at the production call's alignment.
static at::Tensor scratch_like(const at::Tensor& like) {
  const int64_t es = like.element_size();
  const int64_t off = (int64_t)(((uintptr_t)like.data_ptr()) % 256) / es;
  const int64_t span = like.size(0) > 0 ? (like.size(0) - 1) * like.stride(0) + like.size(1) : 0;
  at::Tensor buf = at::empty({span + 256 / es}, like.options());
  return buf.as_strided(like.sizes(), like.strides(), off);
}

static bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  (void)hipStreamIsCapturing(s, &st);
  return st != hipStreamCaptureStatusNone;
}

static float time_algo(hipblasLtHandle_t h, Descs& d, const hipblasLtMatmulAlgo_t& algo, const void* alpha,
                       const void* beta, const void* Bp, const void* Ap, const void* Cp, void* Dp, void* ws, size_t wsz,
                       hipStream_t s, int reps) {
  hipEvent_t e0, e1;
  (void)hipEventCreate(&e0);
  (void)hipEventCreate(&e1);
  // warm-up
  hipblasStatus_t st = hipblasLtMatmul(h, d.op, alpha, Bp, d.A, Ap, d.B, beta, Cp, d.C, Dp, d.D, &algo, ws, wsz, s);
  float ms = -1.f;
  if (st == HIPBLAS_STATUS_SUCCESS) {
    (void)hipEventRecord(e0, s);
    for (int r = 0; r < reps && st == HIPBLAS_STATUS_SUCCESS; ++r)
      st = hipblasLtMatmul(h, d.op, alpha, Bp, d.A, Ap, d.B, beta, Cp, d.C, Dp, d.D, &algo, ws, wsz, s);
    (void)hipEventRecord(e1, s);
    (void)hipEventSynchronize(e1);
    if (st == HIPBLAS_STATUS_SUCCESS) {
      (void)hipEventElapsedTime(&ms, e0, e1);
      ms /= reps;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return ms;
}

// d = alpha * a @ b + beta * (c or d)
void gemm(at::Tensor a, at::Tensor b, at::Tensor d, c10::optional<at::Tensor> c_opt, double alpha_d, double beta_d) {
  TORCH_CHECK(a.is_cuda() && b.is_cuda() && d.is_cuda(), "gemm: GPU tensors required");
  TORCH_CHECK(a.dim() == 2 && b.dim() == 2 && d.dim() == 2, "gemm: 2-D operands required");
  TORCH_CHECK(a.scalar_type() == b.scalar_type(), "gemm: a/b dtype mismatch");
  const int64_t M = a.size(0), K = a.size(1), N = b.size(1);
  TORCH_CHECK(b.size(0) == K && d.size(0) == M && d.size(1) == N, "gemm: shape mismatch");
  TORCH_CHECK(d.stride(1) == 1 && (d.stride(0) >= N || M == 1), "gemm: output must be row-major");
  at::Tensor c = c_opt.has_value() ? *c_opt : d;
  TORCH_CHECK(c.sizes() == d.sizes() && c.stride(1) == 1 && c.scalar_type() == d.scalar_type(), "gemm: bad C");
  if (M == 0 || N == 0) return;
  // column-major: D^T (N x M) = B^T (N x K) * A^T (K x M)
  Problem p{};
  int opA, opB;
  transposed_view(b, &p.rowsA, &p.colsA, &p.lda, &opA);  // hipBLASLt "A" = b^T
  transposed_view(a, &p.rowsB, &p.colsB, &p.ldb, &opB);  // hipBLASLt "B" = a^T
  p.opA = opA;
  p.opB = opB;
  p.m = N;
  p.n = M;
  p.k = K;
  p.ldc = std::max<int64_t>(c.stride(0), N);
  p.ldd = std::max<int64_t>(d.stride(0), N);
  p.ta = dt(a);
  p.tc = dt(d);
  p.beta_nonzero = beta_d != 0.0;
  p.no_sk = no_streamk();
  p.in_place = c.data_ptr() == d.data_ptr();
  p.align = std::min(std::min(ptr_align(a.data_ptr()), ptr_align(b.data_ptr())),
                     std::min(ptr_align(c.data_ptr()), ptr_align(d.data_ptr())));
  const float alpha = (float)alpha_d, beta = (float)beta_d;
  auto& T = Tuner::get();
  hipblasLtHandle_t h = T.handle();
  hipStream_t s = at::hip::getCurrentHIPStream().stream();
  Descs ds;
  make_descs(p, ds);
  const std::string key = p.key();
  Choice ch;
  bool known = T.lookup(key, &ch);
  if (!known) T.log_key(key);
  if (known && !ch.resolved && ch.index >= 0) {
    // a tabled global solution index: resolve it directly
    std::vector<int> idx{ch.index};
    std::vector<hipblasLtMatmulHeuristicResult_t> r;
    size_t wsz = 0;
    if (hipblaslt_ext::getAlgosFromIndex(h, idx, r) == HIPBLAS_STATUS_SUCCESS && !r.empty() &&
        hipblaslt_ext::matmulIsAlgoSupported(h, ds.op, &alpha, ds.A, ds.B, &beta, ds.C, ds.D, r[0].algo, wsz) ==
            HIPBLAS_STATUS_SUCCESS &&
        wsz <= T.max_ws()) {
      ch.algo = r[0].algo;
      ch.ws = wsz;
      ch.resolved = true;
      T.store(key, ch, false);
    } else {
      known = false;  // stale entry (different library build): tune again
    }
  }
  if (!known && T.mode() >= 2 && !capturing(s)) {
    // exhaustive: every library solution for this (ops, dtypes), filtered by support, checked and
    // timed once, the five fastest re-timed.  Each candidate runs on EXACTLY this call's layout:
    // same D / C alignment mod 256 B, and for an in-place accumulation (C == D, the fp32 main_grad
    // of the weight gradients) an aliased C == D scratch holding a copy of the accumulator.  In
    // round 3 candidates were checked out of place (C != D, fresh allocator-aligned D) and some of
    // the picks gave wrong weight gradients in place (profiles/r3_gemm_exhaustive_nosk_wrong.jsonl);
    // tests/test_gemm_exhaustive_gpu.py runs this mode on the in-place TP=8 wgrad shapes.
    std::vector<hipblasLtMatmulHeuristicResult_t> all;
    LT_CHECK(hipblaslt_ext::getAllAlgos(h, hipblaslt_ext::GemmType::HIPBLASLT_GEMM, (hipblasOperation_t)p.opA,
                                        (hipblasOperation_t)p.opB, (hipDataType)p.ta, (hipDataType)p.ta,
                                        (hipDataType)p.tc, (hipDataType)p.tc, HIPBLAS_COMPUTE_32F, all));
    const size_t wsmax = T.max_ws();
    void* wsp = T.workspace(wsmax, s);
    // candidate output: D-layout scratch at D's alignment; C is the same scratch when in place,
    // else the caller's C (read only)
    at::Tensor out_t = scratch_like(d);
    // The accumulator the candidates are validated on is a scratch C of random nonzero values (at
    // C's alignment), never the live one: the first weight-gradient call after zero_grad has
    // main_grad == 0, where a candidate that drops beta * C or mishandles C aliasing D would match.
    at::Tensor c_init;
    if (p.beta_nonzero) {
      c_init = scratch_like(c);
      c_init.normal_();
    }
    void* Dp = out_t.data_ptr();
    const void* Cp = p.in_place ? (const void*)Dp : (p.beta_nonzero ? c_init.data_ptr() : c.data_ptr());
    auto reset = [&]() {
      if (p.beta_nonzero && p.in_place) out_t.copy_(c_init);
    };
    // reference: hipBLASLt's first heuristic choice (the default mode's path), C = c_init, D = a
    // separate buffer
    at::Tensor ref;
    {
      hipblasLtMatmulPreference_t pref;
      LT_CHECK(hipblasLtMatmulPreferenceCreate(&pref));
      uint64_t wm = wsmax;
      LT_CHECK(hipblasLtMatmulPreferenceSetAttribute(pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &wm, sizeof(wm)));
      hipblasLtMatmulHeuristicResult_t r0;
      int got0 = 0;
      LT_CHECK(hipblasLtMatmulAlgoGetHeuristic(h, ds.op, ds.A, ds.B, ds.C, ds.D, pref, 1, &r0, &got0));
      hipblasLtMatmulPreferenceDestroy(pref);
      at::Tensor rbuf = at::empty_like(d);
      const void* rc = p.beta_nonzero ? c_init.data_ptr() : rbuf.data_ptr();
      if (got0 > 0 && hipblasLtMatmul(h, ds.op, &alpha, b.data_ptr(), ds.A, a.data_ptr(), ds.B, &beta, rc, ds.C,
                                      rbuf.data_ptr(), ds.D, &r0.algo, wsp, wsmax, s) == HIPBLAS_STATUS_SUCCESS)
        ref = rbuf.to(at::kFloat, /*non_blocking=*/false, /*copy=*/true);
      if (ref.defined() && !at::isfinite(ref).all().item<bool>()) ref = at::Tensor();   // no usable reference
    }
    const float ref_max = ref.defined() ? ref.abs().max().item<float>() : 0.f;
    // tolerance on the A*B part of the result (a large accumulator must not hide errors in it), plus
    // the output dtype's rounding of the whole value
    float ab_max = ref_max;
    if (ref.defined() && p.beta_nonzero) ab_max = (ref - c_init.to(at::kFloat) * beta).abs().max().item<float>();
    const bool half_out = d.scalar_type() == at::kBFloat16 || d.scalar_type() == at::kHalf;
    const float tol = 2e-2f * ab_max + (half_out ? 8e-3f : 1e-5f) * ref_max + 1e-6f;
    // one untimed run from the reset state, compared with the reference
    auto check = [&](const hipblasLtMatmulAlgo_t& algo) -> bool {
      reset();
      if (hipblasLtMatmul(h, ds.op, &alpha, b.data_ptr(), ds.A, a.data_ptr(), ds.B, &beta, Cp, ds.C, Dp, ds.D, &algo,
                          wsp, wsmax, s) != HIPBLAS_STATUS_SUCCESS)
        return false;
      if (!ref.defined()) return at::isfinite(out_t).all().item<bool>();
      const float err = (out_t.to(at::kFloat) - ref).abs().max().item<float>();   // NaN fails
      return err <= tol;
    };
    std::vector<std::pair<float, int>> timed;
    std::vector<size_t> wss(all.size(), 0);
    auto sweep = [&](bool allow_sk) {
      int tried = 0;
      for (size_t i = 0; i < all.size() && tried < T.max_algos(); ++i) {
        size_t wsz = 0;
        if (hipblaslt_ext::matmulIsAlgoSupported(h, ds.op, &alpha, ds.A, ds.B, &beta, ds.C, ds.D, all[i].algo, wsz) !=
                HIPBLAS_STATUS_SUCCESS ||
            wsz > wsmax || (!allow_sk && is_streamk(h, all[i].algo)))
          continue;
        ++tried;
        wss[i] = wsz;
        if (!check(all[i].algo)) continue;
        const float ms = time_algo(h, ds, all[i].algo, &alpha, &beta, b.data_ptr(), a.data_ptr(), Cp, Dp, wsp, wsmax,
                                   s, 1);
        if (ms > 0.f) timed.emplace_back(ms, (int)i);
      }
    };
    sweep(!p.no_sk);
    if (timed.empty() && p.no_sk) sweep(true);   // no data-parallel solution at all: allow stream-K
    if (!timed.empty()) {  // (nothing passed the check: the heuristic path below decides)
      std::sort(timed.begin(), timed.end());
      int best = -1;
      float best_ms = 1e30f;
      const double flops = 2.0 * M * N * K;
      const int reps = flops > 1e12 ? 5 : (flops > 1e10 ? 10 : 30);
      for (size_t j = 0; j < std::min<size_t>(5, timed.size()); ++j) {
        const int i = timed[j].second;
        float ms = time_algo(h, ds, all[i].algo, &alpha, &beta, b.data_ptr(), a.data_ptr(), Cp, Dp, wsp, wsmax, s,
                             reps);
        if (ms > 0.f && ms < best_ms && check(all[i].algo)) {   // re-checked after the repeated runs
          best_ms = ms;
          best = i;
        }
      }
      if (best >= 0) {
        ch.algo = all[best].algo;
        ch.ws = wss[best];
        ch.ms = best_ms;
        ch.index = hipblaslt_ext::getIndexFromAlgo(all[best].algo);
        ch.resolved = true;
        known = true;
        T.store(key, ch, true);
        if (std::getenv("NXD_GEMM_LOG_CHOICE"))
          std::fprintf(stderr, "[nxd gemm] %s -> %s %.4f ms (exhaustive, %zu timed)\n", key.c_str(),
                       hipblaslt_ext::getKernelNameFromAlgo(h, ch.algo).c_str(), best_ms, timed.size());
      }
    }
  }
  if (!known || !ch.resolved) {
    hipblasLtMatmulPreference_t pref;
    LT_CHECK(hipblasLtMatmulPreferenceCreate(&pref));
    uint64_t wsmax = T.max_ws();
    LT_CHECK(hipblasLtMatmulPreferenceSetAttribute(pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &wsmax,
                                                  sizeof(wsmax)));
    const bool tune = !known && T.mode() >= 1 && !capturing(s);
    // (overlap-safe: a wider heuristic list, the top of which can be all stream-K variants)
    const int want = p.no_sk ? std::max(4 * T.candidates(), 96) : ((tune || known) ? T.candidates() : 1);
    std::vector<hipblasLtMatmulHeuristicResult_t> res(want);
    int got = 0;
    LT_CHECK(hipblasLtMatmulAlgoGetHeuristic(h, ds.op, ds.A, ds.B, ds.C, ds.D, pref, want, res.data(), &got));
    hipblasLtMatmulPreferenceDestroy(pref);
    TORCH_CHECK(got > 0, "gemm: no hipBLASLt solution for ", key);
    // overlap-safe: candidates other than stream-K (all of them if every candidate is stream-K)
    std::vector<char> skip(got, 0);
    if (p.no_sk) {
      int left = 0;   // keep the first candidates() non-stream-K entries
      for (int i = 0; i < got; ++i) {
        skip[i] = is_streamk(h, res[i].algo) || left >= T.candidates();
        left += !skip[i];
      }
      if (left == 0) std::fill(skip.begin(), skip.end(), 0);
    }
    int best = 0;
    while (best + 1 < got && skip[best]) ++best;
    float best_ms = ch.ms;
    if (known) {
      if (ch.pos < got && res[ch.pos].state == HIPBLAS_STATUS_SUCCESS && !skip[ch.pos]) best = ch.pos;
    } else if (tune && got > 1) {
      void* ws = T.workspace(wsmax, s);
      at::Tensor scratch;
      void* Dp = d.data_ptr();
      if (p.beta_nonzero) {  // never accumulate repeatedly into the real output
        scratch = at::empty_like(d);
        Dp = scratch.data_ptr();
      }
      const double flops = 2.0 * M * N * K;
      const int reps = flops > 1e12 ? 3 : (flops > 1e10 ? 8 : 20);
      best = -1;
      std::vector<std::pair<float, int>> first;
      for (int i = 0; i < got; ++i) {
        if (res[i].state != HIPBLAS_STATUS_SUCCESS || res[i].workspaceSize > wsmax || skip[i]) continue;
        float ms = time_algo(h, ds, res[i].algo, &alpha, &beta, b.data_ptr(), a.data_ptr(), c.data_ptr(), Dp, ws,
                             wsmax, s, reps);
        if (ms > 0.f) first.emplace_back(ms, i);
        if (ms > 0.f && (best < 0 || ms < best_ms)) {
          best = i;
          best_ms = ms;
        }
      }
      TORCH_CHECK(best >= 0, "gemm: every candidate failed for ", key);
      // optional (NXD_GEMM_RETIME=n rounds): re-time the leaders round-robin -- one short timing per
      // candidate drifts with the clock the chip holds at that moment, so near-ties are decided by
      // the minimum over interleaved rounds.  1-GPU bench with 3 rounds vs none: 3,031 / 3,032 vs
      // 3,027 / 3,031 ms per step (profiles/r4_gemm_retime_bench_ab.txt), so off by default.
      if (T.retime() > 0 && first.size() > 1) {
        std::sort(first.begin(), first.end());
        const size_t nl = std::min<size_t>(3, first.size());
        std::vector<float> bestr(nl, 1e30f);
        for (int r = 0; r < T.retime(); ++r)
          for (size_t j = 0; j < nl; ++j) {
            const float ms = time_algo(h, ds, res[first[j].second].algo, &alpha, &beta, b.data_ptr(), a.data_ptr(),
                                       c.data_ptr(), Dp, ws, wsmax, s, reps);
            if (ms > 0.f) bestr[j] = std::min(bestr[j], ms);
          }
        size_t w = 0;
        for (size_t j = 1; j < nl; ++j)
          if (bestr[j] < bestr[w]) w = j;
        if (bestr[w] < 1e29f) {
          best = first[w].second;
          best_ms = bestr[w];
        }
      }
    }
    ch.algo = res[best].algo;
    ch.ws = res[best].workspaceSize;
    ch.ms = best_ms;
    ch.pos = best;
    ch.resolved = true;
    T.store(key, ch, tune && got > 1);
    if (std::getenv("NXD_GEMM_LOG_CHOICE"))  // which kernel each new problem runs (stderr)
      std::fprintf(stderr, "[nxd gemm] %s -> %s %.4f ms (pos %d of %d)\n", key.c_str(),
                   hipblaslt_ext::getKernelNameFromAlgo(h, ch.algo).c_str(), best_ms, best, got);
  }
  void* ws = ch.ws ? T.workspace(std::max<size_t>(ch.ws, T.max_ws()), s) : nullptr;
  LT_CHECK(hipblasLtMatmul(h, ds.op, &alpha, b.data_ptr(), ds.A, a.data_ptr(), ds.B, &beta, c.data_ptr(), ds.C,
                           d.data_ptr(), ds.D, &ch.algo, ws, ch.ws ? std::max<size_t>(ch.ws, T.max_ws()) : 0, s));
}

std::vector<std::pair<std::string, float>> gemm_tuned_entries() { return Tuner::get().entries(); }

void gemm_set_no_streamk(int v) { g_no_streamk = v < 0 ? -1 : (v > 0 ? 1 : 0); }
bool gemm_no_streamk() { return no_streamk(); }

// y = act(x w^T) by the kernel of act_gemm.hip
void act_gemm(int64_t act, at::Tensor x, at::Tensor w, at::Tensor y) {
  for (const auto& t : {x, w, y})
    TORCH_CHECK(t.is_cuda() && t.get_device() == x.get_device() && t.scalar_type() == at::kBFloat16 && t.dim() == 2 && t.is_contiguous() &&
                    reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0,
                "act_gemm: contiguous 2-D bf16 on one GPU, 16-byte aligned");
  const int64_t N = y.size(1);
  TORCH_CHECK(w.size(1) == x.size(1) && y.size(0) == x.size(0) && w.size(0) == (act ? N : 2 * N), "act_gemm: sizes");
  const int rc = nxd::act_gemm_launch((int)act, x.data_ptr(), w.data_ptr(), y.data_ptr(), x.size(0), N, x.size(1),
                                      at::hip::getCurrentHIPStream().stream());
  TORCH_CHECK(rc == 0, "act_gemm: failed or not such sizes, ", rc);
}

}  // namespace nxd_gemm

void register_gemm(pybind11::module& m) {
  m.def("gemm", &nxd_gemm::gemm, "d = alpha * a @ b + beta * c (autotuned hipBLASLt)", pybind11::arg("a"),
        pybind11::arg("b"), pybind11::arg("d"), pybind11::arg("c") = pybind11::none(), pybind11::arg("alpha") = 1.0,
        pybind11::arg("beta") = 0.0);
  m.def("act_gemm", &nxd_gemm::act_gemm);
  m.def("gemm_tuned_entries", &nxd_gemm::gemm_tuned_entries);
  m.def("gemm_set_no_streamk", &nxd_gemm::gemm_set_no_streamk, "1: skip stream-K solutions, 0: allow, -1: env");
  m.def("gemm_no_streamk", &nxd_gemm::gemm_no_streamk);
}
