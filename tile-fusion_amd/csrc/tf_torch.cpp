// torch.ops.sw_gcn.* on ROCm tensors: the operators the reference registers for CPU tensors
// (binding-project/main.cpp:133-142), names, argument orders and meanings alike, registered from C++ so that a call
// costs a dispatch and the launches and no Python.  The arithmetic is libtilefusion_hip's, on the tensors' own device
// memory and torch's current stream; torch owns the memory, the stream and the autograd graph.
// tile-fusion_amd/torch_ops.py loads this library and documents the operators.
//
// A training step of the two-layer model on a 3,000-node graph (500 features, 32 hidden, 7 classes) took 332 us with the operators in
// Python, nearly all of it between launches.
#include <ATen/ATen.h>
#include <ATen/SparseCsrTensorUtils.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include <algorithm>
#include <chrono>
#include <list>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "tilefusion_hip.h"

namespace {

using at::Tensor;

void check(tf_status rc) { TORCH_CHECK(rc == TF_OK, "tilefusion status ", (int)rc, ": ", tf_last_error_string()); }

void require_gpu(std::initializer_list<const Tensor *> ts) {
  for (const Tensor *t : ts)
    TORCH_CHECK(t->is_cuda(), "sw_gcn: operands must live on the GPU (a ROCm 'cuda' tensor); this build has no CPU executor");
}

Tensor f32(const Tensor &t) { return t.to(at::kFloat).contiguous(); }

hipStream_t stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// A tensor's memory as a tf_dense for the duration of one call.
class Dense {
 public:
  explicit Dense(const Tensor &t) {
    TORCH_CHECK(t.dim() == 2, "sw_gcn: dense operands are matrices");
    check(tf_dense_wrap_device((int)t.size(0), (int)t.size(1), t.data_ptr<float>(), &h_));
  }
  ~Dense() { tf_dense_free(h_); }
  Dense(const Dense &) = delete;
  Dense &operator=(const Dense &) = delete;
  operator tf_dense *() const { return h_; }

 private:
  tf_dense *h_ = nullptr;
};

// Everything that is built once per adjacency matrix: the host copy of its pattern (the inspector runs on the host), the device CSR,
// schedules per product and widths, its transpose.  Calls that share the schedules' workspaces take turns (Turn).
struct Adjacency : torch::CustomClassHolder {
  std::vector<Tensor> keep;  // a wrapped matrix' arrays stay alive with it
  std::vector<int> Ap, Ai;
  int rows = 0, cols = 0;
  uint64_t hash = 0;
  tf_csr *csr = nullptr;
  std::map<std::pair<int, int>, tf_schedule *> gemm_schedules;  // (K, N)
  std::map<int, tf_schedule *> row_schedules;                   // N, rounded up to a power of two from 32 on
  c10::intrusive_ptr<Adjacency> transposed;                     // null: not built yet, or `symmetric`
  bool symmetric = false;
  std::mutex mutex;
  // the last call that used the workspaces: its stream, and an event behind its work (see Turn); the capture the last captured call
  // belongs to, and an event behind that call in it
  bool used = false;
  hipStream_t last = nullptr;
  hipEvent_t done = nullptr, done_captured = nullptr;
  unsigned long long capture = 0;

  ~Adjacency() override {
    if (done) (void)hipEventDestroy(done);
    if (done_captured) (void)hipEventDestroy(done_captured);
    for (auto &s : gemm_schedules) tf_schedule_free(s.second);
    for (auto &s : row_schedules) tf_schedule_free(s.second);
    tf_csr_free(csr);
  }

  // (the caller holds `mutex`)
  tf_schedule *gemm_schedule(int K, int N) {
    tf_schedule *&s = gemm_schedules[{K, N}];
    if (!s) {
      tf_inspect_opts o{};
      o.struct_size = sizeof(o);
      o.op = TF_OP_GEMM_SPMM;
      o.K = K;
      o.N = N;
      o.pattern_hash = hash;
      check(tf_inspect(rows, cols, Ap.data(), Ai.data(), &o, &s));
    }
    return s;
  }
  tf_schedule *row_schedule(int width) {
    int N = 32;
    while (N < width) N *= 2;
    tf_schedule *&s = row_schedules[N];
    if (!s) check(tf_inspect_spmm(rows, cols, Ap.data(), Ai.data(), N, hash, &s));
    return s;
  }
};
using AdjacencyPtr = c10::intrusive_ptr<Adjacency>;

// A call's turn at an adjacency's schedules: the host calls one after the other, and their work on the device too, whatever streams
// they are on: partial sums, counters and intermediates are the schedule's.
// An event behind every call would do, but costs the stream 3.5 us each (72 us instead of 61 for a training step on 3,000 nodes).  The
// default stream cannot be destroyed or captured, so the event behind its calls is recorded when another stream comes; calls
// on any other stream are followed by an event at once.
// Calls that are being captured are ordered among each other in the graph.  Work from before the capture cannot be waited for
// in a graph, nor can a replay be seen from here: both are the caller's to order, as for all memory a graph uses.
class Turn {
 public:
  Turn(Adjacency &a, hipStream_t st) : lock_(a.mutex), a_(a), st_(st) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    if (st && hipStreamGetCaptureInfo(st, &status, &id) != hipSuccess) (void)hipGetLastError();
    captured_ = status == hipStreamCaptureStatusActive;
    if (captured_) {
      event(a.done_captured);
      if (a.capture == id) check(hipStreamWaitEvent(st, a.done_captured, 0));
      a.capture = 0;
      capture_ = id;
    } else if (a.used && (st || a.last)) {
      event(a.done);
      if (!a.last) check(hipEventRecord(a.done, nullptr));
      check(hipStreamWaitEvent(st, a.done, 0));
    }
    if (!captured_ && st) event(a.done);
  }
  ~Turn() {  // (also when the call failed behind its first launch)
    if (captured_) {
      if (hipEventRecord(a_.done_captured, st_) == hipSuccess) a_.capture = capture_;
    } else {
      if (st_ && hipEventRecord(a_.done, st_) != hipSuccess) (void)hipStreamSynchronize(st_);
      a_.last = st_;
      a_.used = true;
    }
  }
  Turn(const Turn &) = delete;
  Turn &operator=(const Turn &) = delete;

 private:
  static void check(hipError_t e) { TORCH_CHECK(e == hipSuccess, "sw_gcn: ", hipGetErrorString(e)); }
  static void event(hipEvent_t &e) { if (!e) check(hipEventCreateWithFlags(&e, hipEventDisableTiming)); }
  std::lock_guard<std::mutex> lock_;
  Adjacency &a_;
  hipStream_t st_;
  bool captured_ = false;
  unsigned long long capture_ = 0;
};

AdjacencyPtr make_adjacency(const Tensor &adj, const Tensor &crow, const Tensor &col, const Tensor &val) {
  TORCH_CHECK(crow.scalar_type() == at::kInt && col.scalar_type() == at::kInt && val.scalar_type() == at::kFloat,
              "sw_gcn: Adj needs int32 indices and float32 values, as in the reference");
  auto a = c10::make_intrusive<Adjacency>();
  a->keep = {crow, col, val};
  a->rows = (int)adj.size(0);
  a->cols = (int)adj.size(1);
  const Tensor hp = crow.cpu().contiguous(), hi = col.cpu().contiguous();
  a->Ap.assign(hp.data_ptr<int>(), hp.data_ptr<int>() + hp.numel());
  a->Ai.assign(hi.data_ptr<int>(), hi.data_ptr<int>() + hi.numel());
  a->hash = tf_pattern_hash(a->rows, a->Ap.data(), a->Ai.data());
  if (adj.is_cuda()) {
    check(tf_csr_wrap_device(a->rows, a->cols, a->Ap[a->rows], crow.data_ptr<int>(), col.data_ptr<int>(), val.data_ptr<float>(), &a->csr));
    // the device arrays and the host pattern are copies of the same tensors: the executors may check schedules against it
    check(tf_csr_set_pattern_hash(a->csr, a->hash));
    // (the values are read on every call: writes that no version counter shows -- through .data, from another library's kernel,
    // in the replay of a graph -- are honoured)
  }
  return a;
}

// ---- the cache: the last 32 adjacency matrices -------------------------------------------------

using Key = std::tuple<const void *, const void *, const void *, int64_t, int64_t, int64_t, int, int, uint32_t, uint32_t, uint32_t>;
std::mutex g_cache_mutex;
std::list<std::pair<Key, AdjacencyPtr>> g_cache;  // most recent first
constexpr size_t kCacheSize = 32;

AdjacencyPtr adjacency_of(const Tensor &adj) {
  TORCH_CHECK(adj.layout() == at::kSparseCsr, "sw_gcn: Adj must be a sparse CSR tensor");
  const auto *impl = at::sparse_csr::get_sparse_csr_impl(adj);
  const Tensor &crow = impl->compressed_indices(), &col = impl->plain_indices(), &val = impl->values();
  // the version counters change with every in-place update of the tensors: a cached host pattern,
  // schedule or transpose is never used for values or indices that were changed afterwards
  const Key key{crow.data_ptr(), col.data_ptr(), val.data_ptr(), adj.size(0), adj.size(1), val.numel(), (int)adj.device().type(), adj.device().index(),
                (uint32_t)crow._version(), (uint32_t)col._version(), (uint32_t)val._version()};
  std::lock_guard<std::mutex> lock(g_cache_mutex);
  for (auto it = g_cache.begin(); it != g_cache.end(); ++it)
    if (it->first == key) {
      if (it != g_cache.begin()) g_cache.splice(g_cache.begin(), g_cache, it);
      return it->second;
    }
  AdjacencyPtr a = make_adjacency(adj, crow.detach(), col.detach(), val.detach());
  g_cache.emplace_front(key, a);
  if (g_cache.size() > kCacheSize) g_cache.pop_back();
  return a;
}

void clear_cache() {
  std::lock_guard<std::mutex> lock(g_cache_mutex);
  g_cache.clear();
}

// out = the transpose of the rows x cols matrix (p, i, x), rows sorted by column.
void transpose_csr(int rows, int cols, const int *p, const int *i, const float *x, std::vector<int> &tp, std::vector<int> &ti, std::vector<float> &tx) {
  const int nnz = p[rows];
  tp.assign(cols + 1, 0);
  ti.resize(nnz);
  tx.resize(nnz);
  for (int k = 0; k < nnz; ++k) ++tp[i[k] + 1];
  for (int c = 0; c < cols; ++c) tp[c + 1] += tp[c];
  std::vector<int> at(tp.begin(), tp.end() - 1);
  for (int r = 0; r < rows; ++r)
    for (int k = p[r]; k < p[r + 1]; ++k) {
      const int q = at[i[k]]++;
      ti[q] = r;
      tx[q] = x[k];
    }
}

// The transpose as another adjacency (the same one when symmetric), built when first asked for.
AdjacencyPtr transpose_of(const AdjacencyPtr &a) {
  std::lock_guard<std::mutex> lock(a->mutex);
  if (a->symmetric) return a;
  if (a->transposed) return a->transposed;
  const Tensor hv = a->keep[2].cpu().contiguous();
  auto t = c10::make_intrusive<Adjacency>();
  t->rows = a->cols;
  t->cols = a->rows;
  std::vector<float> tx;
  transpose_csr(a->rows, a->cols, a->Ap.data(), a->Ai.data(), hv.data_ptr<float>(), t->Ap, t->Ai, tx);
  if (a->Ap == t->Ap) {
    // (equal row lengths: compare the entries, of the matrix with its rows sorted where they are not)
    std::vector<int> sp, si;
    std::vector<float> sx;
    const int *ai = a->Ai.data();
    const float *ax = hv.data_ptr<float>();
    bool sorted = true;
    for (int r = 0; r < a->rows && sorted; ++r)
      for (int k = a->Ap[r] + 1; k < a->Ap[r + 1]; ++k) sorted = sorted && ai[k - 1] <= ai[k];
    if (!sorted) {
      transpose_csr(t->rows, t->cols, t->Ap.data(), t->Ai.data(), tx.data(), sp, si, sx);
      ai = si.data();
      ax = sx.data();
    }
    if (std::equal(t->Ai.begin(), t->Ai.end(), ai) && std::equal(tx.begin(), tx.end(), ax)) {
      a->symmetric = true;
      return a;
    }
  }
  check(tf_csr_upload(t->rows, t->cols, t->Ap.data(), t->Ai.data(), tx.data(), &t->csr));
  // an identity of its own for its schedules, in the place of another pass over the pattern
  t->hash = a->hash ^ 0x7472616E73706F73ull;
  if (!t->hash) t->hash = 1;
  check(tf_csr_set_pattern_hash(t->csr, t->hash));
  a->transposed = t;
  return t;
}

// ---- the products ------------------------------------------------------------------------------

// a * (X * W), W in x out, or out x in (w_t) as torch stores a layer's weights
Tensor gemm_spmm(Adjacency &a, const Tensor &x_, const Tensor &w_, bool w_t, bool relu) {
  require_gpu({&x_, &w_});
  const Tensor x = f32(x_), w = f32(w_);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2, "sw_gcn: dense operands are matrices");
  const int64_t K = x.size(1), N = w.size(w_t ? 0 : 1);
  TORCH_CHECK(a.cols == x.size(0) && w.size(w_t ? 1 : 0) == K, "sw_gcn: shapes do not chain: Adj (", a.rows, ", ", a.cols, "), Feature ", x.sizes(), ", weight ", w.sizes());
  c10::OptionalDeviceGuard guard(x.device());
  Tensor out = at::empty({a.rows, N}, x.options());
  Dense xb(x), wb(w), ob(out);
  const Turn turn(a, stream_of(x));
  check(tf_gemm_spmm(a.csr, xb, wb, ob, a.gemm_schedule((int)K, (int)N), (w_t ? TF_C_TRANSPOSED : 0u) | (relu ? TF_RELU : 0u), stream_of(x)));
  return out;
}

// a * X
Tensor spmm(Adjacency &a, const Tensor &x_) {
  require_gpu({&x_});
  const Tensor x = f32(x_);
  c10::OptionalDeviceGuard guard(x.device());
  Tensor out = at::empty({a.rows, x.size(1)}, x.options());
  Dense xb(x), ob(out);
  const Turn turn(a, stream_of(x));
  check(tf_spmm_scheduled(a.csr, xb, ob, a.row_schedule((int)x.size(1)), 0, stream_of(x)));
  return out;
}

// t * W, W stored as the second factor is read; zero where `mask` is zero or less
Tensor gemm(const Tensor &t, const Tensor &w_, const Tensor *mask) {
  const Tensor w = f32(w_);
  c10::OptionalDeviceGuard guard(t.device());
  Tensor out = at::empty({t.size(0), w.size(1)}, t.options());
  Dense tb(t), wb(w), ob(out);
  if (mask) {
    Dense mb(*mask);
    check(tf_gemm_ex(tb, wb, ob, mb, 0, stream_of(t)));
  } else {
    check(tf_gemm_ex(tb, wb, ob, nullptr, 0, stream_of(t)));
  }
  return out;
}

// t^T * x: the gradient of a layer's weights (out x in), t = A^T times the gradient of the layer's output
struct WeightGrad {
  Tensor t, x, out, ws;
  WeightGrad(const Tensor &t_, const Tensor &x_) : t(t_), x(f32(x_)) {
    const int M = (int)t.size(0), N = (int)t.size(1), K = (int)x.size(1);
    out = at::empty({N, K}, t.options());
    const int64_t floats = (int64_t)(tf_weight_grad_workspace(M, N, K) / sizeof(float));
    if (floats > 0) ws = at::empty({floats}, t.options());
  }
  float *workspace() const { return ws.defined() ? ws.data_ptr<float>() : nullptr; }
};
Tensor weight_grad(const Tensor &t, const Tensor &x) {
  c10::OptionalDeviceGuard guard(t.device());
  const WeightGrad w(t, x);
  Dense tb(w.t), xb(w.x), ob(w.out);
  check(tf_weight_grad(tb, xb, ob, w.workspace(), stream_of(t)));
  return w.out;
}
// both layers' at once
void weight_grads(const Tensor &t1, const Tensor &x1, const Tensor &t2, const Tensor &x2, Tensor *g1, Tensor *g2) {
  c10::OptionalDeviceGuard guard(t1.device());
  const WeightGrad a(t1, x1), b(t2, x2);
  Dense ta(a.t), xa(a.x), oa(a.out), tb(b.t), xb(b.x), ob(b.out);
  check(tf_weight_grad_pair(ta, xa, oa, a.workspace(), tb, xb, ob, b.workspace(), stream_of(t1)));
  *g1 = a.out;
  *g2 = b.out;
}

// ---- autograd ------------------------------------------------------------------------------------

using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;

c10::IValue hold(const AdjacencyPtr &a) { return c10::IValue::make_capsule(a); }
AdjacencyPtr held(const c10::IValue &v) { return c10::static_intrusive_pointer_cast<Adjacency>(v.toCapsule()); }

// The gradients of D = A (X W^T) for X and W.  Both come out of T = A^T G: grad X = T W, grad W = T^T X, so that the
// sparse product, the dearer half, is done once and at the layer's output width.
void layer_gradients(const AdjacencyPtr &at, const Tensor &G, const Tensor &x, const Tensor &w, bool want_x, bool want_w, Tensor *gx, Tensor *gw) {
  if (want_x && !want_w) {
    *gx = gemm_spmm(*at, G, w, false, false);
    return;
  }
  if (!want_w) return;
  const Tensor T = spmm(*at, G);
  if (want_x) *gx = gemm(T, w, nullptr);
  *gw = weight_grad(T, x);
}

// FusedGeMMSpMM / FusedGeMMSpMMROAdj (binding-project/src/Functions.cpp:1248-1268, 1192-1246) and UnFusedGeMMSpMM:
// forward Adj @ (Feature @ Weight^T) with Weight [out, in]; backward for Feature and Weight.
struct Layer : public torch::autograd::Function<Layer> {
  static Tensor forward(AutogradContext *ctx, const AdjacencyPtr &a, const Tensor &feature, const Tensor &weight, bool fused) {
    ctx->saved_data["adj"] = hold(a);
    ctx->save_for_backward({feature, weight});
    if (fused) return gemm_spmm(*a, feature, weight, true, false);
    require_gpu({&feature, &weight});
    return spmm(*a, at::mm(feature, weight.t()));  // the two products as separate launches, the intermediate in HBM
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    Tensor gx, gw;
    layer_gradients(transpose_of(held(ctx->saved_data["adj"])), grads[0], saved[0], saved[1], ctx->needs_input_grad(0), ctx->needs_input_grad(1), &gx, &gw);
    return {Tensor(), gx, gw, Tensor()};
  }
};

// Two layers with a ReLU between; the hidden layer is kept for the backward pass, where the step back through the
// ReLU is part of the product that leads to it.
struct TwoLayers : public torch::autograd::Function<TwoLayers> {
  static Tensor forward(AutogradContext *ctx, const AdjacencyPtr &a, const Tensor &x, const Tensor &w1, const Tensor &w2) {
    const Tensor hidden = gemm_spmm(*a, x, w1, true, true);
    ctx->saved_data["adj"] = hold(a);
    ctx->save_for_backward({x, w1, w2, hidden});
    return gemm_spmm(*a, hidden, w2, true, false);
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &w1 = saved[1], &w2 = saved[2], &hidden = saved[3];
    const bool want_x = ctx->needs_input_grad(0), want_1 = ctx->needs_input_grad(1), want_2 = ctx->needs_input_grad(2);
    const AdjacencyPtr at = transpose_of(held(ctx->saved_data["adj"]));
    Tensor gx, g1, g2;
    const Tensor T = spmm(*at, grads[0]);
    if (want_1 && want_2) {
      const Tensor T1 = spmm(*at, gemm(T, w2, &hidden));
      if (want_x) gx = gemm(T1, w1, nullptr);
      weight_grads(T1, x, T, hidden, &g1, &g2);
      return {Tensor(), gx, g1, g2};
    }
    if (want_2) g2 = weight_grad(T, hidden);
    if (want_x || want_1) layer_gradients(at, gemm(T, w2, &hidden), x, w1, want_x, want_1, &gx, &g1);
    return {Tensor(), gx, g1, g2};
  }
};

// ---- the operators (names and argument orders of main.cpp:5-27) --------------------------------

// The schedule in the binding project's layout (Functions.cpp:588-622): LevelPtr[3]; MixPtr[2p] = start of a partition's
// first-op ids, MixPtr[2p+1] = start of its second-op ids, MixPtr[2P] = end; Partition = the ids.
std::vector<Tensor> schedule_tensors(const AdjacencyPtr &a, int K, int N) {
  std::lock_guard<std::mutex> lock(a->mutex);
  tf_schedule_view v{};
  v.struct_size = sizeof(v);
  check(tf_schedule_get_view(a->gemm_schedule(K, N), &v));
  const int P = v.ptr1[2];
  Tensor level = at::empty({3}, at::kInt), mix = at::empty({2 * (int64_t)P + 2}, at::kInt), ids = at::empty({v.n_id}, at::kInt);
  std::copy(v.ptr1, v.ptr1 + 3, level.data_ptr<int>());
  std::copy(v.id, v.id + v.n_id, ids.data_ptr<int>());
  int *m = mix.data_ptr<int>();
  for (int p = 0; p < P; ++p) {
    m[2 * p] = v.ptr2[p];
    m[2 * p + 1] = v.ker_begin[2 * p];
  }
  m[2 * P] = m[2 * P + 1] = v.ptr2[P];
  return {level, mix, ids};
}

std::vector<Tensor> inspect(const Tensor &adj, int64_t) { return schedule_tensors(adjacency_of(adj), 64, 64); }

std::vector<Tensor> inspect_vt_ro(const Tensor &adj, int64_t in_dim, int64_t out_dim, int64_t, int64_t) {
  return schedule_tensors(adjacency_of(adj), (int)in_dim, (int)out_dim);
}

// Weight is [in, out] here, not transposed (main.cpp:76-103); returns (out, seconds).
std::vector<Tensor> execute_fused(const Tensor &adj, const Tensor &weight, const Tensor &feature, const Tensor &, const Tensor &, const Tensor &, int64_t) {
  require_gpu({&adj, &weight, &feature});
  check(tf_device_synchronize());
  const auto t0 = std::chrono::steady_clock::now();
  const Tensor out = gemm_spmm(*adjacency_of(adj), feature, weight, false, false);
  check(tf_device_synchronize());
  return {out, at::scalar_tensor(std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count(), at::TensorOptions(at::kFloat))};
}

Tensor fused_layer(const Tensor &adj, const Tensor &feature, const Tensor &weight, at::TensorList, int64_t) {
  require_gpu({&adj, &feature, &weight});
  return Layer::apply(adjacency_of(adj), feature, weight, true);
}

Tensor fused_layer_vt_ro(const Tensor &adj, const Tensor &feature, const Tensor &weight, at::TensorList schedule, int64_t threads, int64_t) {
  return fused_layer(adj, feature, weight, schedule, threads);
}

// ForwardCachingAF: (Adj @ Feature), computed once by the caller, times Weight^T.
Tensor cached_layer(const Tensor &af, const Tensor &weight, int64_t) { return at::mm(af, weight.t()); }

Tensor unfused_layer(const Tensor &adj, const Tensor &feature, const Tensor &weight, int64_t) {
  require_gpu({&adj, &feature, &weight});
  return Layer::apply(adjacency_of(adj), feature, weight, false);
}

// Adj @ (relu(Adj @ (Feature @ Weight1^T)) @ Weight2^T), weights [out, in]: the forward of the reference's end-to-end model
// (gcn-e2e-training/FusedGCNModule.py:14-18) and the composition its unregistered fusedGCN
// (binding-project/src/Functions.cpp:228-290) stands for.
Tensor fused_gcn(const Tensor &adj, const Tensor &feature, const Tensor &weight1, const Tensor &weight2, int64_t) {
  require_gpu({&adj, &feature, &weight1, &weight2});
  const AdjacencyPtr a = adjacency_of(adj);
  if (at::GradMode::is_enabled() && (feature.requires_grad() || weight1.requires_grad() || weight2.requires_grad()))
    return TwoLayers::apply(a, feature, weight1, weight2);
  const Tensor x = f32(feature), w1 = f32(weight1), w2 = f32(weight2);
  TORCH_CHECK(x.dim() == 2 && w1.dim() == 2 && w2.dim() == 2, "sw_gcn: dense operands are matrices");
  const int64_t K = x.size(1), H = w1.size(0), N = w2.size(0);
  TORCH_CHECK(a->rows == a->cols && a->cols == x.size(0) && w1.size(1) == K && w2.size(1) == H, "sw_gcn: shapes do not chain: Adj (", a->rows, ", ",
              a->cols, "), Feature ", x.sizes(), ", weights ", w1.sizes(), ", ", w2.sizes());
  c10::OptionalDeviceGuard guard(x.device());
  Tensor out = at::empty({a->rows, N}, x.options());
  Dense xb(x), b1(w1), b2(w2), ob(out);
  const Turn turn(*a, stream_of(x));
  tf_schedule *s1 = a->gemm_schedule((int)K, (int)H), *s2 = a->gemm_schedule((int)H, (int)N);
  check(tf_gcn_two_layers(a->csr, xb, b1, b2, ob, s1, s2, nullptr, TF_RELU | TF_C_TRANSPOSED, stream_of(x)));
  return out;
}

}  // namespace

TORCH_LIBRARY(sw_gcn, m) {
  m.def("inspect(Tensor Adj, int MTileSize) -> Tensor[]", &inspect);
  m.def("inspect_vt_ro(Tensor Adj, int InDim, int OutDim, int CacheSize, int NumThreads) -> Tensor[]", &inspect_vt_ro);
  m.def("executeFusedGeMMSpMM(Tensor Adj, Tensor Weight, Tensor Feature, Tensor LevelPtr, Tensor MixPtr, Tensor Partition, int NumThreads) -> Tensor[]", &execute_fused);
  m.def("fusedGeMMSpMM(Tensor Adj, Tensor Feature, Tensor Weight, Tensor[] Schedule, int NumThreads) -> Tensor", &fused_layer);
  m.def("fusedGeMMSpMM_vt_ro(Tensor Adj, Tensor Feature, Tensor Weight, Tensor[] Schedule, int NumThreads, int MaxTileSize) -> Tensor", &fused_layer_vt_ro);
  m.def("geMMSpMM_f_bw(Tensor Adj, Tensor Feature, Tensor Weight, Tensor[] Schedule, int NumThreads) -> Tensor", &fused_layer);
  m.def("cachedSpMMGeMM(Tensor AF, Tensor Weight, int NumThreads) -> Tensor", &cached_layer);
  m.def("unfused_gcn_forward(Tensor Adj, Tensor Feature, Tensor Weight, int NumThreads) -> Tensor", &unfused_layer);
  m.def("fusedGCN(Tensor Adj, Tensor Feature, Tensor Weight1, Tensor Weight2, int NumThreads) -> Tensor", &fused_gcn);
}

extern "C" void sw_gcn_clear_cache() { clear_cache(); }
