// C ABI of libtilefusion_hip: error channel, device objects, executors.
// Compiled by hipcc together with tf_inspector.cpp and tf_kernels.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <new>

#include "tf_internal.h"
#include "tf_rows.h"

// ---- handles ---------------------------------------------------------------------

struct tf_csr {
  int M = 0, N = 0, nnz = 0;
  int *p = nullptr, *i = nullptr;
  float *x = nullptr;
  bool owns = false;
  // > 0 for an uploaded matrix: its device arrays never change, so work derived from its values
  // (the regrouped values of column-partitioned long rows) is done once per schedule
  unsigned long long serial = 0;
  uint64_t hash = 0;  // tf_pattern_hash of the host arrays it was uploaded from (0: unknown, wrapped)
};

struct tf_dense {
  int M = 0, N = 0;
  float *d = nullptr;
  bool owns = false;
};

namespace tf {

struct DeviceSchedule {
  int device = -1;
  char *arena = nullptr;  // one allocation for the lists and the workspace, which the pointers below name parts of
  TileDesc *tiles = nullptr;
  int *fused_ids = nullptr;
  int *win = nullptr;
  int *rem_rows = nullptr;
  int *zero_rows = nullptr;
  int *plain_rows = nullptr;
  int *step_begin = nullptr;  // streamed GeMM-SpMM: per launched tile, first entry in step_ptr
  int *step_ptr = nullptr;
  int *fused_rec = nullptr;
  LongChunk *long_chunks = nullptr;
  LongRow *long_rows = nullptr;  // the rows that partial sums are added up for: of several chunks, or of segments
  int n_long_rows = 0, n_big_rows = 0;  // of segments: those with groups of them come first
  int *chunk_long = nullptr;     // per chunk: which of long_rows it belongs to, -1 when it is its row's only one
  unsigned *arrived = nullptr;   // per row of several chunks: how many of them are done
  LongRow *seg_groups = nullptr;
  float *inter = nullptr;    // M x N intermediate, only if some tile writes back
  float *spare = nullptr;    // ... one of its own, for runs over a stencil that are asked once for what they are not for
  float *partial = nullptr;  // n_long_chunks (or segments) x N
  int *seg_ptr = nullptr, *seg_src = nullptr, *seg_col = nullptr, *lrow_seg = nullptr;  // column-partitioned long rows
  float *seg_val = nullptr;  // A's values in the order of the regrouped entries
  unsigned long long seg_val_serial = 0;  // the uploaded matrix they were taken from (0: none)
  // the short remainder rows stored in the order of the row list: row pointers, columns, where each value (rem_first: each
  // row's first) comes from in A's array, and the values themselves (of the matrix rem_val_serial that does not change)
  int *rem_ptr = nullptr, *rem_col = nullptr, *rem_src = nullptr, *rem_first = nullptr;
  bool rem_first_known = false;
  float *rem_val = nullptr;
  unsigned long long rem_val_serial = 0;
  Tile2 *l2_tiles = nullptr; // two-layer tiles
  float *hidden = nullptr;   // tf_gcn_two_layers: the first layer's output, L x K of this (second-layer) schedule
  size_t hidden_floats = 0;
  float *Bpad = nullptr;     // M x K' copy of B, zero-padded, when K is not a multiple of 8
  float *Cpad = nullptr;     // K' x N copy of C, zero-padded or from its transpose
  float *Cpanel = nullptr;   // K' x N and L x N: one column panel of C (zero-padded) and of D, when the caller's width is
  float *Dpanel = nullptr;   // not one the kernels take (user_N != N)
  // marching runs: the schedule's lists, and the ELL rows with the operands' values filled in
  int *m_runs = nullptr, *m_row_ptr = nullptr, *m_load_ptr = nullptr, *m_load = nullptr, *m_row_out = nullptr;
  int *m_ell_off = nullptr, *m_ell_src = nullptr, *m_ell = nullptr;
  float *m_trash = nullptr;  // a row in global memory that takes the stores of lane groups without a row
  unsigned long long m_serial_a = 0, m_serial_b = 0;  // the uploaded matrices the values were taken from (0: none)
  // A second stream of the same priority for kernels that may run beside the caller's stream (the
  // hot long-row segments beside the rest of the GEMM), with the events that fork it off and join it.
  hipStream_t side = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
  // per-launch timing, when tf_schedule_set_profiling switched it on
  int prof_n = 0;
  const char *prof_name[TF_PROFILE_MAX] = {};
  hipEvent_t prof_ev[TF_PROFILE_MAX][2] = {};
};

// launchers in tf_kernels.hip
hipError_t launch_fused_spmm_spmm(const TileDesc *, int, const int *, const int *, const int *,
                                  const float *, const float *, const int *, const int *,
                                  const float *, float *, float *, int, int, int, hipStream_t);
hipError_t launch_fused_spmm_spmm_window(const TileDesc *, const int *, int, const int *, const int *,
                                         const int *, const float *, const float *, float *, int, int,
                                         int, int, hipStream_t);
hipError_t launch_fused_spmm_spmm_window64(const TileDesc *, const int *, int, const int *, const int *,
                                           const float *, int, const float *, const int *, const int *,
                                           const float *, int, float *, int, int, int, int, hipStream_t);
hipError_t launch_spmm_rows(RowsArgs, const RowsHow &, hipStream_t);
hipError_t launch_spmm_gemm(RowsArgs, const RowsHow &, const float *, int, int, const GemmOut &, hipStream_t);
hipError_t launch_gemm_any(const float *, int, const float *, int, float *, int, const int *, int, int, int, int, const GemmOut &, int, hipStream_t);
WeightGradTask plan_weight_grad(int, int, int, int);
hipError_t launch_weight_grads(const WeightGradTask &, const WeightGradTask *, hipStream_t);
hipError_t launch_gather_values(const int *, const float *, float *, int, hipStream_t);
hipError_t launch_fused_box(BoxArgs, int, hipStream_t);
hipError_t launch_fused_star(BoxArgs, int, hipStream_t);
hipError_t launch_march_fill(const int *, const int *, const float *, const float *, int *, size_t, hipStream_t);
hipError_t launch_fused_spmm_spmm_march(const int *, int, const int *, const int *, const int *, const int *, const int *,
                                        const float *, float *, float *, int, int, int, int, int, int, int, hipStream_t);
hipError_t launch_seg_reduce(const LongRow *, int, int, const LongRow *, int, const int *, const float *, float *, int, int, int, int, hipStream_t);
hipError_t launch_fused_gemm_spmm(const TileDesc *, int, const int *, const float *, const float *,
                                  int, int, const int *, const int *, const float *, float *,
                                  float *, int, int, int, int, int, hipStream_t);
hipError_t launch_fused_gemm_spmm_stream(const TileDesc *, int, const int *, const int *, const int *,
                                         const float *, const float *, int, int, int, const int *,
                                         const float *, float *, float *, int, int, hipStream_t, int relu_in = 0);
hipError_t launch_fill(float *, size_t, float, hipStream_t);
hipError_t launch_pad(const float *, int, int, float *, int, int, hipStream_t);
hipError_t launch_transpose_pad(const float *, int, int, int, int, float *, int, int, hipStream_t);
hipError_t launch_copy_cols(const float *, int, int, int, int, float *, int, int, int, int, int, hipStream_t);
hipError_t launch_relu(float *, size_t, hipStream_t);
hipError_t launch_fused_gcn2(const Tile2 *, int, const float *, const float *, const float *, int, int, int, const int *, const int *,
                             const float *, float *, int, int, int, hipStream_t);
hipError_t launch_xcd_probe(int *, int, hipStream_t);
hipError_t launch_issue_probe(float *, int, int, int, int, hipStream_t);

// An intermediate larger than the 256 MB last-level cache is gone from it before its readers
// come: such rows leave through streaming stores.
inline int inter_streams(const tf_schedule *s) {
  return (size_t)s->M * s->opts.N * sizeof(float) > ((size_t)256 << 20) ? 1 : 0;
}

static thread_local char g_err[512] = "";

tf_status fail(tf_status code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

static tf_status hip_fail(hipError_t e, const char *what) {
  return fail(e == hipErrorOutOfMemory ? TF_ENOMEM : TF_EHIP, "%s: %s", what, hipGetErrorString(e));
}

#define TF_HIP(call)                                         \
  do {                                                       \
    hipError_t e_ = (call);                                  \
    if (e_ != hipSuccess) return tf::hip_fail(e_, #call);    \
  } while (0)

int default_compute_units() {
  static std::atomic<int> known[64];  // per device, once asked for
  int dev = 0, cu = 0;
  if (hipGetDevice(&dev) == hipSuccess) {
    if (dev >= 0 && dev < 64 && (cu = known[dev].load(std::memory_order_relaxed)) > 0) return cu;
    if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cu > 0) {
      if (dev >= 0 && dev < 64) known[dev].store(cu, std::memory_order_relaxed);
      return cu;
    }
  }
  (void)hipGetLastError();
  return 256;
}

void release_device_schedule(DeviceSchedule *d) {
  if (!d) return;
  (void)hipFree(d->arena); (void)hipFree(d->hidden); (void)hipFree(d->spare);
  if (d->side) (void)hipStreamDestroy(d->side);
  if (d->fork) (void)hipEventDestroy(d->fork);
  if (d->join) (void)hipEventDestroy(d->join);
  for (auto &pair : d->prof_ev)
    for (hipEvent_t e : pair)
      if (e) (void)hipEventDestroy(e);
  delete d;
}

// The parts of a schedule's arena: lists to be copied there and workspace to be reserved, collected first and then made with
// one allocation; lists of up to 64 KB, which come first, travel in one copy.  (An allocation, its release and a small copy
// each cost tens of microseconds: a schedule has up to thirty arrays.)
class ArenaParts {
 public:
  template <class T> void list(const std::vector<T> &v, T **out) {
    *out = nullptr;
    if (!v.empty()) add(v.data(), v.size() * sizeof(T), out);
  }
  template <class T> void reserve(size_t n, T **out) { add(nullptr, std::max<size_t>(n, 1) * sizeof(T), out); }
  tf_status make(char **arena) {
    std::stable_partition(parts_.begin(), parts_.end(), [](const Part &p) { return small(p); });
    size_t total = 0, packed = 0;
    for (Part &p : parts_) {  // (the large ones start where an allocation of their own would: at a page)
      const size_t align = p.bytes >= ((size_t)2 << 20) ? (size_t)2 << 20 : 256;
      p.at = (total + align - 1) / align * align;
      total = p.at + p.bytes;
      if (small(p)) packed = total;
    }
    if (total == 0) return TF_OK;
    TF_HIP(hipMalloc(reinterpret_cast<void **>(arena), total));
    std::vector<char> stage(packed);
    for (const Part &p : parts_) {
      *p.out = *arena + p.at;
      if (small(p)) std::memcpy(stage.data() + p.at, p.data, p.bytes);
    }
    if (packed > 0) TF_HIP(hipMemcpy(*arena, stage.data(), packed, hipMemcpyHostToDevice));
    for (const Part &p : parts_)
      if (p.data && !small(p)) TF_HIP(hipMemcpy(*arena + p.at, p.data, p.bytes, hipMemcpyHostToDevice));
    return TF_OK;
  }

 private:
  struct Part { const void *data; size_t bytes, at; void **out; };
  static bool small(const Part &p) { return p.data && p.bytes <= 65536; }
  template <class T> void add(const void *data, size_t bytes, T **out) { parts_.push_back({data, bytes, 0, reinterpret_cast<void **>(out)}); }
  std::vector<Part> parts_;
};

// A GeMM-SpMM schedule in which nothing fuses is a GEMM into the intermediate and row products out of it, for which K
// and N are what the caller has.  (Tiles take K in steps of 8 and N in steps of 32: padded copies, column panels.)
static bool untiled(const tf_schedule *s) { return s->opts.op == TF_OP_GEMM_SPMM && (s->launch_tiles.empty() || s->two_passes); }
// Floats from one row of the intermediate to the next: a multiple of 4, so that every lane's columns of a row are one
// aligned load, and whole cache lines where the row kernel then works in column slices (slices_for in tf_rows.hip).
static int inter_ld(const tf_schedule *s) {
  if (!untiled(s) && !s->two_passes && !s->box) return s->opts.N;
  const int N = s->user_N;
  return N > 96 && N < 128 && s->M >= 16000 && s->M <= 131072 ? 128 : (N + 3) / 4 * 4;
}

// Device copies of the schedule arrays and the workspace, made on first use.
static tf_status ensure_device(tf_schedule *s) {
  static std::mutex mu;
  std::lock_guard<std::mutex> lock(mu);
  int dev = 0;
  TF_HIP(hipGetDevice(&dev));
  if (s->dev) {
    if (s->dev->device != dev)
      return fail(TF_ESCHEDULE, "schedule was uploaded to device %d, current device is %d", s->dev->device, dev);
    return TF_OK;
  }
  auto *d = new (std::nothrow) DeviceSchedule();
  if (!d) return fail(TF_ENOMEM, "out of host memory");
  d->device = dev;
  ArenaParts parts;
  const std::vector<float> trash(64, 0.f);
  std::vector<LongChunk> chunks;
  std::vector<LongRow> summed;  // the rows that partial sums are added up for
  std::vector<int> chunk_long;
  std::vector<unsigned> arrived;
  if (s->two_passes) {  // (the lists are the other schedule's)
    parts.reserve(s->spmm_first ? (size_t)s->L * s->user_K : (size_t)s->M * inter_ld(s), &d->inter);
    parts.list(s->l2_tiles, &d->l2_tiles);
  } else if (s->box) {  // no lists; the calls that the runs are not for are two products
    if (s->box_room) parts.reserve((size_t)s->M * inter_ld(s), &d->inter);
  } else if (s->march) {  // nothing but the run lists is needed on the device
    parts.list(s->march_runs, &d->m_runs);
    parts.list(s->march_row_ptr, &d->m_row_ptr);
    parts.list(s->march_load_ptr, &d->m_load_ptr);
    parts.list(s->march_load, &d->m_load);
    parts.list(s->march_row_out, &d->m_row_out);
    parts.list(s->march_ell_off, &d->m_ell_off);
    parts.list(s->march_ell_src, &d->m_ell_src);
    parts.reserve(s->march_ell_off.size() * 2, &d->m_ell);
    parts.list(trash, &d->m_trash);
  } else {
    parts.list(s->launch_tiles, &d->tiles);
    parts.list(s->l2_tiles, &d->l2_tiles);
    parts.list(s->fused_ids, &d->fused_ids);
    parts.list(s->win, &d->win);
    parts.list(s->rem_rows, &d->rem_rows);
    parts.list(s->zero_rows, &d->zero_rows);
    parts.list(s->plain_rows, &d->plain_rows);
    parts.list(s->launch_step, &d->step_begin);
    parts.list(s->step_ptr, &d->step_ptr);
    parts.list(s->fused_rec, &d->fused_rec);
    if (!s->rem_ptr.empty()) {
      parts.list(s->rem_ptr, &d->rem_ptr);
      parts.list(s->rem_col, &d->rem_col);
      parts.list(s->rem_src, &d->rem_src);
      parts.reserve(s->rem_src.size(), &d->rem_val);
      parts.reserve(s->rem_rows.size(), &d->rem_first);
    }
    const size_t N = (size_t)std::max(s->opts.N, s->user_N);
    size_t slots = 0;  // partial sums
    if (!s->long_chunks.empty()) {
      // The chunk of a row that has no other goes straight to the row of the result (slot -1); only rows of several
      // chunks need partial sums and the launch that adds them up.
      chunks = s->long_chunks;
      for (const LongRow &lr : s->long_rows) {
        if (lr.count == 1) { chunks[lr.first].slot = -1; continue; }
        summed.push_back({lr.row, (int)slots, lr.count, 0});
        for (int c = 0; c < lr.count; ++c) chunks[lr.first + c].slot = (int)slots++;
      }
      // longest first: what starts last should end soon
      std::stable_sort(chunks.begin(), chunks.end(), [](const LongChunk &a, const LongChunk &b) { return a.k_end - a.k_begin > b.k_end - b.k_begin; });
      parts.list(chunks, &d->long_chunks);
      std::vector<int> of_slot(slots);
      for (size_t r = 0; r < summed.size(); ++r) std::fill_n(of_slot.begin() + summed[r].first, summed[r].count, (int)r);
      for (const LongChunk &c : chunks) chunk_long.push_back(c.slot < 0 ? -1 : of_slot[c.slot]);
      parts.list(chunk_long, &d->chunk_long);
      arrived.assign(summed.size(), 0);
      parts.list(arrived, &d->arrived);
    } else {
      summed = s->long_rows;
      const int n_seg = (int)s->seg_ptr.size() - 1;
      d->n_big_rows = (int)(std::stable_partition(summed.begin(), summed.end(), [&](const LongRow &lr) { return lr.count > 0 && s->lrow_seg[lr.first] >= n_seg; }) - summed.begin());
    }
    parts.list(summed, &d->long_rows);
    d->n_long_rows = (int)summed.size();
    if (s->long_part) {
      parts.list(s->seg_ptr, &d->seg_ptr);
      parts.list(s->seg_src, &d->seg_src);
      parts.list(s->seg_col, &d->seg_col);
      parts.list(s->lrow_seg, &d->lrow_seg);
      parts.list(s->seg_groups, &d->seg_groups);
      parts.reserve(s->seg_src.size(), &d->seg_val);
      slots = s->seg_ptr.size() - 1;
    }
    if (slots > 0) parts.reserve(slots * N, &d->partial);
    if (s->n_writeback_rows > 0) parts.reserve((size_t)s->M * inter_ld(s), &d->inter);
    const bool tiled = s->opts.op == TF_OP_GEMM_SPMM && !s->launch_tiles.empty();
    if (tiled && s->user_N != s->opts.N) {
      parts.reserve((size_t)s->opts.K * s->opts.N, &d->Cpanel);
      parts.reserve((size_t)s->L * s->opts.N, &d->Dpanel);
    }
    if (tiled && s->user_K != s->opts.K) parts.reserve((size_t)s->M * s->opts.K, &d->Bpad);
    // (also where K needs no padding: any call may come with TF_C_TRANSPOSED, and a captured one cannot allocate)
    if (tiled && s->user_N == s->opts.N) parts.reserve((size_t)s->opts.K * s->opts.N, &d->Cpad);
  }
  tf_status rc = parts.make(&d->arena);
  if (!rc && s->long_part && s->plain_hot > 0) {
    hipError_t e = hipStreamCreateWithFlags(&d->side, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&d->fork, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&d->join, hipEventDisableTiming);
    if (e != hipSuccess) rc = hip_fail(e, "hipStreamCreate(side stream)");
  }
  if (rc) { release_device_schedule(d); return rc; }
  s->dev = d;
  return TF_OK;
}

// Timing of one launch (or group of launches) of an executor call: events around it on its stream.
static hipError_t prof_begin(tf_schedule *s, const char *name, hipStream_t st) {
  DeviceSchedule *d = s->dev;
  if (!s->profiling || d->prof_n >= TF_PROFILE_MAX) return hipSuccess;
  const int n = d->prof_n;
  for (int q = 0; q < 2; ++q)
    if (!d->prof_ev[n][q]) {
      hipError_t e = hipEventCreate(&d->prof_ev[n][q]);
      if (e != hipSuccess) return e;
    }
  d->prof_name[n] = name;
  return hipEventRecord(d->prof_ev[n][0], st);
}
static hipError_t prof_end(tf_schedule *s, hipStream_t st) {
  DeviceSchedule *d = s->dev;
  if (!s->profiling || d->prof_n >= TF_PROFILE_MAX) return hipSuccess;
  return hipEventRecord(d->prof_ev[d->prof_n++][1], st);
}
#define TF_PHASE(sched, name, st, call)        \
  do {                                         \
    TF_HIP(tf::prof_begin(sched, name, st));   \
    TF_HIP(call);                              \
    TF_HIP(tf::prof_end(sched, st));           \
  } while (0)

static bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// What to remember as the matrix whose values a call on `st` puts in a schedule's order: none (0) when the call is being captured, for
// nothing is written before the graph is launched, if it ever is.
static unsigned long long written_now(hipStream_t st, unsigned long long serial) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (st && hipStreamIsCapturing(st, &status) != hipSuccess) (void)hipGetLastError();
  return status == hipStreamCaptureStatusNone ? serial : 0;
}

// The hot segments of column-partitioned long rows: segments of partition p are worked on by the
// workgroups that land on XCD p.  The values in the order of the regrouped entries -- what the
// reference's reordered adjacency (createReorderedAdj, GCN_Single_Layer_SP_Demo_Utils.h:618-653)
// is to its executors -- are built on the first call with an uploaded matrix and kept; a wrapped
// matrix can change between calls, so its values are regrouped every time.
// ensure_segment_values fills the values of ALL segments, hot and cold, so it must run on a stream
// that both the hot and the cold launch are ordered after: the caller's, before a second stream forks.
static tf_status ensure_segment_values(const tf_csr *A, tf_schedule *s, hipStream_t st) {
  DeviceSchedule *d = s->dev;
  if (A->serial != 0 && d->seg_val_serial == A->serial) return TF_OK;
  TF_PHASE(s, "gather_values_kernel", st, launch_gather_values(d->seg_src, A->x, d->seg_val, (int)s->seg_src.size(), st));
  d->seg_val_serial = written_now(st, A->serial);
  return TF_OK;
}
// What the row products of a call read and write: T (row stride ldt) the intermediate or, for a rows-only schedule, the
// operand itself; N columns.
struct Remainder {
  const float *T;
  int ldt, N, rows;  // rows of T
  float *D;
  int accumulate, relu;
  int streaming = 1;  // D is not read again by this library
  int ldd = 0;        // floats from one row of D to the next (0: N)
};
static tf_status run_hot_segments(tf_schedule *s, const Remainder &r, hipStream_t st) {
  DeviceSchedule *d = s->dev;
  RowsArgs a;
  a.n_rows = 8 * s->seg_per_xcd;
  a.Ap = d->seg_ptr; a.Ai = d->seg_col; a.Ax = d->seg_val;
  a.X = r.T; a.ldx = r.ldt; a.x_rows = r.rows; a.Y = d->partial; a.ldy = r.N; a.N = r.N;
  a.streaming = 1;
  RowsHow how;
  how.xcd_chunk_rows = -1;
  TF_PHASE(s, "spmm_rows_kernel (hot long-row segments)", st, launch_spmm_rows(a, how, st));
  return TF_OK;
}

// The row kernel's operands for the remainder rows and the chunks of the long ones.
static tf_status remainder_rows(const tf_csr *A, tf_schedule *s, const Remainder &r, hipStream_t st, RowsArgs &a, RowsHow &how) {
  DeviceSchedule *d = s->dev;
  const int N = r.N, ldd = r.ldd > 0 ? r.ldd : r.N;
  a.n_rows = (int)s->rem_rows.size();
  a.Ap = A->p; a.Ai = A->i; a.Ax = A->x;
  a.X = r.T; a.ldx = r.ldt; a.x_rows = r.rows; a.Y = r.D; a.ldy = ldd; a.N = N;
  a.accumulate = r.accumulate; a.relu = r.relu; a.streaming = r.streaming;
  how.xcd_chunk_rows = s->row_deal;
  how.spread_entries = s->rem_sweep ? A->nnz : 0;
  a.zero_rows = d->zero_rows;
  a.n_zero = r.accumulate && !r.relu ? 0 : (int)s->zero_rows.size();  // (D += 0 needs nothing)
  a.chunks = d->long_chunks;
  a.n_chunks = (unsigned)s->long_chunks.size();
  a.chunk_Ai = A->i; a.chunk_Ax = A->x; a.partial = d->partial;
  a.chunk_long = d->chunk_long; a.long_rows = d->long_rows; a.arrived = d->arrived;
  if (!s->rem_rows.empty() && !s->rem_ptr.empty()) {
    // The rows in the order of the list, columns side by side -- the reference's reordered adjacency
    // (createReorderedAdj, GCN_Single_Layer_SP_Demo_Utils.h:618-653; executor at
    // GCN_Layer_MKL_Forward_Utils.h:294-373).  The values of a matrix whose device arrays never change are copied into that
    // order on the first call and kept; those of any other are read in place, where they are on every call (a layer's two products
    // of 100,000 rows of 11 entries, N = 64: 171 us, 165 with kept values, 177 with a copy per call).
    a.rows = d->rem_rows;
    a.Ap = d->rem_ptr; a.Ai = d->rem_col;
    if (A->serial == 0) {
      if (!d->rem_first_known) {  // (a part of the pattern: the same for every matrix the schedule is run on)
        TF_PHASE(s, "gather_values_kernel", st,
                 launch_gather_values(d->rem_rows, reinterpret_cast<const float *>(A->p), reinterpret_cast<float *>(d->rem_first), a.n_rows, st));
        d->rem_first_known = written_now(st, 1) != 0;
      }
      a.val_first = d->rem_first;
    } else {
      if (d->rem_val_serial != A->serial) {
        TF_PHASE(s, "gather_values_kernel", st, launch_gather_values(d->rem_src, A->x, d->rem_val, (int)s->rem_src.size(), st));
        d->rem_val_serial = written_now(st, A->serial);
      }
      a.Ax = d->rem_val;
    }
    a.compact = 1;
    how.flagged = s->rem_flagged ? 1 : 0;
  } else if (!s->rem_identity) {
    a.rows = d->rem_rows;
  }
  return TF_OK;
}

// Second-op rows that no tile fused: served from the intermediate in HBM.  hot_on_side: the hot
// long-row segments were launched on the side stream already and are joined here.
static tf_status run_remainder(const tf_csr *A, tf_schedule *s, const Remainder &r, bool hot_on_side, hipStream_t st) {
  DeviceSchedule *d = s->dev;
  const int N = r.N, ldd = r.ldd > 0 ? r.ldd : r.N;
  if (d->partial && N > std::max(s->opts.N, s->user_N))
    return fail(TF_ESCHEDULE, "the schedule's partial sums have %d columns, the product has %d", std::max(s->opts.N, s->user_N), N);
  RowsArgs a;
  RowsHow how;
  if (tf_status rc = remainder_rows(A, s, r, st, a, how)) return rc;
  // one launch, the long rows' workgroups first
  if (a.n_rows > 0 || a.n_chunks > 0)
    TF_PHASE(s, sweep_for(a, how).LPR > 0 ? "sweep_rows_kernel" : a.n_chunks > 0 ? "spmm_rows_kernel (short and long remainder rows)" : "spmm_rows_kernel (short remainder rows)", st,
             launch_spmm_rows(a, how, st));
  if (s->long_part) {
    const int n_hot = 8 * s->seg_per_xcd, n_seg = (int)s->seg_ptr.size() - 1;
    if (!hot_on_side) {
      if (tf_status rc = ensure_segment_values(A, s, st)) return rc;
      if (tf_status rc = run_hot_segments(s, r, st)) return rc;
    }
    RowsArgs c;
    c.n_rows = n_seg - n_hot;
    c.Ap = d->seg_ptr + n_hot; c.Ai = d->seg_col; c.Ax = d->seg_val;
    c.X = r.T; c.ldx = r.ldt; c.x_rows = r.rows; c.Y = d->partial + (size_t)n_hot * N; c.ldy = N; c.N = N;
    c.streaming = 1;
    TF_PHASE(s, "spmm_rows_kernel (cold long-row segments)", st, launch_spmm_rows(c, RowsHow(), st));
    if (hot_on_side) TF_HIP(hipStreamWaitEvent(st, d->join, 0));
    TF_PHASE(s, "long_seg_reduce_kernel", st,
             launch_seg_reduce(d->long_rows, d->n_long_rows, d->n_big_rows, d->seg_groups, n_seg, d->lrow_seg, d->partial, r.D, ldd, N, r.accumulate, r.relu, st));
  }
  return TF_OK;
}

}  // namespace tf

using tf::fail;

// The fixed scratch array of tf_spmm_spmm_noalloc (further down) and its per-device address.
namespace {

constexpr size_t kScratchFloats = (size_t)8 << 20;  // 32 MiB: e.g. 65,536 intermediate rows of 128 columns
static __device__ __align__(256) float scratch[kScratchFloats];

constexpr int kMaxDevices = 64;
float *g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_mu;

// The device address of the current device's copy of `scratch`, looked up once per device.
// (In host code the array's name is only a handle for this lookup, never an address.)
tf_status scratch_of_current_device(float **out) {
  int dev = 0;
  TF_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return fail(TF_EUNSUPPORTED, "device ordinal %d is beyond the %d this library keeps scratch addresses for", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    TF_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return fail(TF_EHIP, "hipGetSymbolAddress returned a null address for the scratch array");
    g_scratch_ptr[dev] = static_cast<float *>(p);
  }
  *out = g_scratch_ptr[dev];
  return TF_OK;
}

}  // namespace


// ---- errors, device, streams -----------------------------------------------------

extern "C" const char *tf_last_error_string(void) { return tf::g_err; }
extern "C" const char *tf_version(void) { return "0.1"; }

extern "C" tf_status tf_device_init(int device, tf_device_info *info) {
  int count = 0;
  hipError_t e = hipGetDeviceCount(&count);
  if (e != hipSuccess || count <= 0) {
    (void)hipGetLastError();
    return fail(TF_EHIP, "no HIP device available (%s)", e == hipSuccess ? "count is 0" : hipGetErrorString(e));
  }
  if (device < 0 || device >= count) return fail(TF_EINVAL, "device %d out of range (have %d)", device, count);
  TF_HIP(hipSetDevice(device));
  {
    float *unused = nullptr;
    if (tf_status rc = scratch_of_current_device(&unused)) return rc;
  }
  if (info) {
    if (info->struct_size < TF_SIZE_THROUGH(tf_device_info, xcd_round_robin))  // before any work is done for it
      return fail(TF_EINVAL, "tf_device_init: info->struct_size is %zu, the struct's first version has %zu bytes (set it to sizeof(tf_device_info))",
                  info->struct_size, TF_SIZE_THROUGH(tf_device_info, xcd_round_robin));
    hipDeviceProp_t p;
    TF_HIP(hipGetDeviceProperties(&p, device));
    tf_device_info full;
    std::memset(&full, 0, sizeof(full));
    tf_device_info *const caller = info;
    info = &full;
    info->device = device;
    info->compute_units = p.multiProcessorCount;
    info->xcds = 8;
    info->lds_bytes_per_block = (int)p.sharedMemPerBlock;
    int optin = 0;
    if (hipDeviceGetAttribute(&optin, hipDeviceAttributeSharedMemPerBlockOptin, device) == hipSuccess && optin > info->lds_bytes_per_block)
      info->lds_bytes_per_block = optin;
    (void)hipGetLastError();
    info->wavefront = p.warpSize;
    info->clock_khz = p.clockRate;
    info->hbm_bytes = p.totalGlobalMem;
    std::snprintf(info->arch, sizeof(info->arch), "%s", p.gcnArchName);
    // Workgroup b of a launch is expected on XCD b mod 8: checked once here, on 64 workgroups.
    info->xcd_round_robin = -1;
    int *probe = nullptr, host[64];
    if (hipMalloc(reinterpret_cast<void **>(&probe), sizeof(host)) == hipSuccess) {
      if (tf::launch_xcd_probe(probe, 64, nullptr) == hipSuccess &&
          hipMemcpy(host, probe, sizeof(host), hipMemcpyDeviceToHost) == hipSuccess) {
        bool ok = true;
        for (int b = 0; b < 64 && ok; ++b) ok = host[b] == host[b % info->xcds];
        for (int a = 0; a < info->xcds && ok; ++a)
          for (int b = a + 1; b < info->xcds && ok; ++b) ok = host[a] != host[b];
        info->xcd_round_robin = ok ? 1 : 0;
      }
      (void)hipFree(probe);
    }
    (void)hipGetLastError();
    return tf::emit_out("tf_device_init", caller, full, TF_SIZE_THROUGH(tf_device_info, xcd_round_robin));
  }
  return TF_OK;
}

extern "C" tf_status tf_device_synchronize(void) {
  TF_HIP(hipDeviceSynchronize());
  return TF_OK;
}

extern "C" tf_status tf_calibrate_issue(int role_older, int role_younger, int iters, float *ms) {
  if (!ms || iters <= 0 || iters > (1 << 20) || role_older < 0 || role_older > 3 || role_younger < 0 || role_younger > 3)
    return fail(TF_EINVAL, "tf_calibrate_issue: roles are 0 .. 3, iters 1 .. 2^20");
  float *out = nullptr;
  TF_HIP(hipMalloc(reinterpret_cast<void **>(&out), 512 * sizeof(float)));
  hipEvent_t e0 = nullptr, e1 = nullptr;
  hipError_t err = hipEventCreate(&e0);
  if (err == hipSuccess) err = hipEventCreate(&e1);
  const int cus = tf::default_compute_units(), reps = 5;
  if (err == hipSuccess) err = tf::launch_issue_probe(out, cus, iters, role_older, role_younger, nullptr);  // warm-up
  if (err == hipSuccess) err = hipEventRecord(e0, nullptr);
  for (int r = 0; r < reps && err == hipSuccess; ++r) err = tf::launch_issue_probe(out, cus, iters, role_older, role_younger, nullptr);
  if (err == hipSuccess) err = hipEventRecord(e1, nullptr);
  if (err == hipSuccess) err = hipEventSynchronize(e1);
  float t = 0.f;
  if (err == hipSuccess) err = hipEventElapsedTime(&t, e0, e1);
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  (void)hipFree(out);
  TF_HIP(err);
  *ms = t / reps;
  return TF_OK;
}

extern "C" tf_status tf_stream_create(void **stream) {
  if (!stream) return fail(TF_EINVAL, "tf_stream_create: null");
  hipStream_t s;
  TF_HIP(hipStreamCreate(&s));
  *stream = s;
  return TF_OK;
}
extern "C" tf_status tf_stream_destroy(void *stream) {
  if (stream) TF_HIP(hipStreamDestroy(static_cast<hipStream_t>(stream)));
  return TF_OK;
}
extern "C" tf_status tf_stream_synchronize(void *stream) {
  TF_HIP(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
  return TF_OK;
}
extern "C" tf_status tf_event_create(void **event) {
  if (!event) return fail(TF_EINVAL, "tf_event_create: null");
  hipEvent_t e;
  TF_HIP(hipEventCreate(&e));
  *event = e;
  return TF_OK;
}
extern "C" tf_status tf_event_destroy(void *event) {
  if (event) TF_HIP(hipEventDestroy(static_cast<hipEvent_t>(event)));
  return TF_OK;
}
extern "C" tf_status tf_event_record(void *event, void *stream) {
  TF_HIP(hipEventRecord(static_cast<hipEvent_t>(event), static_cast<hipStream_t>(stream)));
  return TF_OK;
}
extern "C" tf_status tf_event_synchronize(void *event) {
  TF_HIP(hipEventSynchronize(static_cast<hipEvent_t>(event)));
  return TF_OK;
}
extern "C" tf_status tf_event_elapsed_ms(void *start, void *stop, float *ms) {
  if (!ms) return fail(TF_EINVAL, "tf_event_elapsed_ms: null");
  TF_HIP(hipEventElapsedTime(ms, static_cast<hipEvent_t>(start), static_cast<hipEvent_t>(stop)));
  return TF_OK;
}

// a matrix whose device arrays never change has a number of its own
static std::atomic<unsigned long long> g_next_serial{1};

// ---- operands ----------------------------------------------------------------------

extern "C" tf_status tf_csr_upload(int M, int N, const int *Ap, const int *Ai, const float *Ax,
                                   tf_csr **out) {
  if (!out) return fail(TF_EINVAL, "tf_csr_upload: out is null");
  *out = nullptr;
  if (M <= 0 || N <= 0 || !Ap) return fail(TF_EINVAL, "tf_csr_upload: bad M/N/Ap");
  if (Ap[0] != 0) return fail(TF_EINVAL, "tf_csr_upload: Ap[0] != 0");
  for (int r = 0; r < M; ++r)
    if (Ap[r + 1] < Ap[r]) return fail(TF_EINVAL, "tf_csr_upload: Ap not monotone at row %d", r);
  const int nnz = Ap[M];
  if (nnz > 0 && (!Ai || !Ax)) return fail(TF_EINVAL, "tf_csr_upload: Ai/Ax null");
  for (int k = 0; k < nnz; ++k)
    if (Ai[k] < 0 || Ai[k] >= N) return fail(TF_EINVAL, "tf_csr_upload: column %d out of range at entry %d", Ai[k], k);
  auto *a = new (std::nothrow) tf_csr();
  if (!a) return fail(TF_ENOMEM, "out of host memory");
  a->M = M; a->N = N; a->nnz = nnz; a->owns = true;
  a->serial = g_next_serial.fetch_add(1);
  a->hash = tf_pattern_hash(M, Ap, Ai);
  hipError_t e = hipMalloc(reinterpret_cast<void **>(&a->p), (size_t)(M + 1) * sizeof(int));
  if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void **>(&a->i), (size_t)std::max(nnz, 1) * sizeof(int));
  if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void **>(&a->x), (size_t)std::max(nnz, 1) * sizeof(float));
  if (e == hipSuccess) e = hipMemcpy(a->p, Ap, (size_t)(M + 1) * sizeof(int), hipMemcpyHostToDevice);
  if (e == hipSuccess && nnz > 0) e = hipMemcpy(a->i, Ai, (size_t)nnz * sizeof(int), hipMemcpyHostToDevice);
  if (e == hipSuccess && nnz > 0) e = hipMemcpy(a->x, Ax, (size_t)nnz * sizeof(float), hipMemcpyHostToDevice);
  if (e != hipSuccess) { tf_csr_free(a); return tf::hip_fail(e, "tf_csr_upload"); }
  *out = a;
  return TF_OK;
}

extern "C" tf_status tf_csr_wrap_device(int M, int N, int nnz, const int *dAp, const int *dAi,
                                        const float *dAx, tf_csr **out) {
  if (!out) return fail(TF_EINVAL, "tf_csr_wrap_device: out is null");
  *out = nullptr;
  if (M <= 0 || N <= 0 || nnz < 0 || !dAp || (nnz > 0 && (!dAi || !dAx)))
    return fail(TF_EINVAL, "tf_csr_wrap_device: bad argument");
  auto *a = new (std::nothrow) tf_csr();
  if (!a) return fail(TF_ENOMEM, "out of host memory");
  a->M = M; a->N = N; a->nnz = nnz; a->owns = false;
  a->p = const_cast<int *>(dAp); a->i = const_cast<int *>(dAi); a->x = const_cast<float *>(dAx);
  *out = a;
  return TF_OK;
}

extern "C" tf_status tf_csr_set_pattern_hash(tf_csr *a, uint64_t hash) {
  if (!a) return fail(TF_EINVAL, "tf_csr_set_pattern_hash: null argument");
  a->hash = hash;
  return TF_OK;
}

extern "C" tf_status tf_csr_set_constant(tf_csr *a) {
  if (!a) return fail(TF_EINVAL, "tf_csr_set_constant: null argument");
  a->serial = g_next_serial.fetch_add(1);
  return TF_OK;
}

extern "C" void tf_csr_free(tf_csr *a) {
  if (!a) return;
  if (a->owns) { (void)hipFree(a->p); (void)hipFree(a->i); (void)hipFree(a->x); }
  delete a;
}

extern "C" tf_status tf_dense_alloc(int M, int N, tf_dense **out) {
  if (!out) return fail(TF_EINVAL, "tf_dense_alloc: out is null");
  *out = nullptr;
  if (M <= 0 || N <= 0) return fail(TF_EINVAL, "tf_dense_alloc: bad shape %d x %d", M, N);
  auto *d = new (std::nothrow) tf_dense();
  if (!d) return fail(TF_ENOMEM, "out of host memory");
  d->M = M; d->N = N; d->owns = true;
  hipError_t e = hipMalloc(reinterpret_cast<void **>(&d->d), (size_t)M * N * sizeof(float));
  if (e != hipSuccess) { delete d; return tf::hip_fail(e, "tf_dense_alloc"); }
  *out = d;
  return TF_OK;
}

extern "C" tf_status tf_dense_upload(int M, int N, const float *host, tf_dense **out) {
  if (!host) return fail(TF_EINVAL, "tf_dense_upload: host is null");
  tf_status rc = tf_dense_alloc(M, N, out);
  if (rc) return rc;
  hipError_t e = hipMemcpy((*out)->d, host, (size_t)M * N * sizeof(float), hipMemcpyHostToDevice);
  if (e != hipSuccess) { tf_dense_free(*out); *out = nullptr; return tf::hip_fail(e, "tf_dense_upload"); }
  return TF_OK;
}

extern "C" tf_status tf_dense_wrap_device(int M, int N, float *dptr, tf_dense **out) {
  if (!out) return fail(TF_EINVAL, "tf_dense_wrap_device: out is null");
  *out = nullptr;
  if (M <= 0 || N <= 0 || !dptr) return fail(TF_EINVAL, "tf_dense_wrap_device: bad argument");
  if (!tf::aligned16(dptr)) return fail(TF_EINVAL, "tf_dense_wrap_device: pointer must be 16-byte aligned");
  auto *d = new (std::nothrow) tf_dense();
  if (!d) return fail(TF_ENOMEM, "out of host memory");
  d->M = M; d->N = N; d->d = dptr; d->owns = false;
  *out = d;
  return TF_OK;
}

extern "C" tf_status tf_dense_download(const tf_dense *d, float *host) {
  if (!d || !host) return fail(TF_EINVAL, "tf_dense_download: null argument");
  TF_HIP(hipMemcpy(host, d->d, (size_t)d->M * d->N * sizeof(float), hipMemcpyDeviceToHost));
  return TF_OK;
}

extern "C" tf_status tf_dense_fill(tf_dense *d, float value, void *stream) {
  if (!d) return fail(TF_EINVAL, "tf_dense_fill: null argument");
  TF_HIP(tf::launch_fill(d->d, (size_t)d->M * d->N, value, static_cast<hipStream_t>(stream)));
  return TF_OK;
}

extern "C" tf_status tf_dense_copy(tf_dense *dst, const tf_dense *src, void *stream) {
  if (!dst || !src) return fail(TF_EINVAL, "tf_dense_copy: null argument");
  if (dst->M != src->M || dst->N != src->N)
    return fail(TF_EINVAL, "tf_dense_copy: shapes differ (%d x %d and %d x %d)", dst->M, dst->N, src->M, src->N);
  TF_HIP(hipMemcpyAsync(dst->d, src->d, (size_t)src->M * src->N * sizeof(float), hipMemcpyDeviceToDevice,
                        static_cast<hipStream_t>(stream)));
  return TF_OK;
}

extern "C" float *tf_dense_device_ptr(const tf_dense *d) { return d ? d->d : nullptr; }

extern "C" void tf_dense_free(tf_dense *d) {
  if (!d) return;
  if (d->owns) (void)hipFree(d->d);
  delete d;
}

// ---- executors -----------------------------------------------------------------------

static tf_status check_pattern(const char *who, const tf_csr *A, const tf_schedule *s) {
  if (A->M != s->L || A->N != s->M || A->nnz != s->nnz)
    return fail(TF_ESCHEDULE, "%s: schedule was built for a %d x %d pattern with %lld entries, A is %d x %d with %d",
                who, s->L, s->M, s->nnz, A->M, A->N, A->nnz);
  if (A->hash && A->hash != s->pattern_hash)
    return fail(TF_ESCHEDULE, "%s: A has the shape and entry count the schedule was built for, but another sparsity pattern", who);
  return TF_OK;
}

static tf_status check_common(const char *who, const tf_csr *A, const tf_dense *C, const tf_dense *D,
                              const tf_schedule *s, int op, bool c_transposed = false) {
  if (!A || !C || !D || !s) return fail(TF_EINVAL, "%s: null argument", who);
  if (s->rows_only) return fail(TF_ESCHEDULE, "%s: the schedule is one of tf_inspect_spmm", who);
  if (s->opts.op != op) return fail(TF_ESCHEDULE, "%s: schedule was built for the other operation", who);
  if (tf_status rc = check_pattern(who, A, s)) return rc;
  const int cn = c_transposed ? C->M : C->N;
  if (cn != s->user_N || D->N != s->user_N)
    return fail(TF_ESCHEDULE, "%s: schedule was built for N = %d, C has %d and D has %d columns", who, s->user_N, cn, D->N);
  if (D->M != A->M) return fail(TF_EINVAL, "%s: D has %d rows, A has %d", who, D->M, A->M);
  return TF_OK;
}

// Y = A X for every row of A in order.
static tf::RowsArgs all_rows(const tf_csr *A, const float *X, float *Y, int N) {
  tf::RowsArgs a;
  a.n_rows = A->M;
  a.Ap = A->p; a.Ai = A->i; a.Ax = A->x;
  a.X = X; a.ldx = N; a.x_rows = A->N; a.Y = Y; a.ldy = N; a.N = N;
  return a;
}

// What runs over a stencil are not for, in the schedule's stead: both products row by row through an intermediate in HBM, the same sums in the same order.
static tf_status box_as_two_products(const tf_csr *A, const tf_csr *B, const tf_dense *C, tf_dense *D, tf_schedule *s, int acc, hipStream_t st) {
  tf::DeviceSchedule *d = s->dev;
  const int N = s->opts.N, ldt = tf::inter_ld(s);
  if (!d->inter) {
    TF_HIP(hipMalloc(reinterpret_cast<void **>(&d->spare), (size_t)s->M * ldt * sizeof(float)));
    d->inter = d->spare;
  }
  tf::RowsArgs first = all_rows(B, C->d, d->inter, N), second = all_rows(A, d->inter, D->d, N);
  first.ldy = second.ldx = ldt;
  first.streaming = tf::inter_streams(s);
  second.streaming = 1;
  second.accumulate = acc;
  tf::RowsHow how;
  how.xcd_chunk_rows = s->row_deal;
  TF_PHASE(s, "spmm_rows_kernel (intermediate rows)", st, tf::launch_spmm_rows(first, tf::RowsHow(), st));
  TF_PHASE(s, "spmm_rows_kernel (second-op rows)", st, tf::launch_spmm_rows(second, how, st));
  return TF_OK;
}

extern "C" tf_status tf_spmm_spmm(const tf_csr *A, const tf_csr *B, const tf_dense *C, tf_dense *D,
                                  tf_schedule *s, unsigned flags, void *stream) {
  tf_status rc = check_common("tf_spmm_spmm", A, C, D, s, TF_OP_SPMM_SPMM);
  if (rc) return rc;
  if (!B) return fail(TF_EINVAL, "tf_spmm_spmm: B is null");
  if (B->M != A->N) return fail(TF_EINVAL, "tf_spmm_spmm: B has %d rows, A has %d columns", B->M, A->N);
  if (C->M != B->N) return fail(TF_EINVAL, "tf_spmm_spmm: C has %d rows, B has %d columns", C->M, B->N);
  rc = tf::ensure_device(s);
  if (rc) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int acc = (flags & TF_ACCUMULATE) ? 1 : 0;
  tf::DeviceSchedule *d = s->dev;
  d->prof_n = 0;
  const int n_launch = (int)s->launch_tiles.size();
  const bool other_inner = s->march && (B->nnz != s->inner_nnz || B->N != s->opts.inner_cols || (B->hash && B->hash != s->inner_hash));
  if (other_inner && !s->box_beside)
    return fail(TF_ESCHEDULE, "tf_spmm_spmm: the schedule's runs were built on another inner pattern than B's");
  if (s->two_passes) {
    tf_schedule *rows = s->two_passes;
    if ((rc = tf::ensure_device(rows))) return rc;
    rows->profiling = s->profiling;
    rows->dev->prof_n = 0;
    const int N = s->opts.N, ldt = tf::inter_ld(s);
    // (the lists hold A's columns: they serve B when it has A's pattern)
    const bool same = B == A || (B->p == A->p && B->i == A->i && B->x == A->x) || (B->hash && B->hash == s->pattern_hash);
    if (same) {
      tf::Remainder first{C->d, N, N, C->M, d->inter, 0, 0, tf::inter_streams(s)};
      first.ldd = ldt;
      rc = tf::run_remainder(B, rows, first, false, st);
    } else {
      tf::RowsArgs a = all_rows(B, C->d, d->inter, N);
      a.ldy = ldt;
      a.streaming = tf::inter_streams(s);
      TF_PHASE(rows, "spmm_rows_kernel (intermediate rows)", st, tf::launch_spmm_rows(a, tf::RowsHow(), st));
    }
    if (rc) return rc;
    return tf::run_remainder(A, rows, tf::Remainder{d->inter, ldt, N, s->M, D->d, acc, 0}, false, st);
  }
  if (s->box) {
    // (a wrapped matrix without a hash may have any pattern; who has runs that always were runs has given B the inner one)
    const bool unknown_inner = s->box_room && !B->hash && !(B->p == A->p && B->i == A->i);
    // (a run reads what is around its points in C while others store theirs in D; two products have read C when D is stored)
    const bool in_place = D->d < C->d + (size_t)C->M * C->N && C->d < D->d + (size_t)D->M * D->N;
    if (other_inner || unknown_inner || in_place) return box_as_two_products(A, B, C, D, s, acc, st);
    tf::BoxArgs a = s->box_runs;
    a.Ax = A->x; a.Bx = B->x; a.C = C->d; a.D = D->d;
    a.val_bytes = (unsigned)A->nnz * 4;
    if (a.star) TF_PHASE(s, "fused_star_kernel", st, tf::launch_fused_star(a, acc, st));
    else TF_PHASE(s, "fused_box_kernel", st, tf::launch_fused_box(a, acc, st));
    return TF_OK;
  }
  if (s->march) {
    // The values in the order of the runs' ELL rows (the reference's reordered adjacency,
    // createReorderedAdj, GCN_Single_Layer_SP_Demo_Utils.h:618-653): filled in on the first call with
    // uploaded matrices, whose device arrays never change, and on every call with wrapped ones.
    const bool have = A->serial != 0 && B->serial != 0 && d->m_serial_a == A->serial && d->m_serial_b == B->serial;
    if (!have) {
      TF_PHASE(s, "march_fill_kernel", st, tf::launch_march_fill(d->m_ell_off, d->m_ell_src, A->x, B->x, d->m_ell, s->march_ell_off.size(), st));
      d->m_serial_a = tf::written_now(st, A->serial);
      d->m_serial_b = tf::written_now(st, B->serial);
    }
    TF_PHASE(s, "fused_spmm_spmm_march_kernel", st,
             tf::launch_fused_spmm_spmm_march(d->m_runs, (int)s->march_runs.size() / 2, d->m_row_ptr, d->m_load_ptr, d->m_load,
                                              d->m_row_out, d->m_ell, C->d, D->d, d->m_trash, s->opts.N, s->lds_bytes, s->march_tpg,
                                              s->march_dpg, s->march_lpg, s->march_width, acc, st));
    return TF_OK;
  }
  if (s->windowed) {
    if (B->nnz != s->inner_nnz || B->N != s->opts.inner_cols)
      return fail(TF_ESCHEDULE, "tf_spmm_spmm: schedule was built for an inner pattern with %lld entries and %d columns, B has %d and %d",
                  s->inner_nnz, s->opts.inner_cols, B->nnz, B->N);
    // the windowed kernels turn B's columns into LDS offsets inside the tile's window of C: another
    // pattern would read outside it
    if (B->hash && B->hash != s->inner_hash)
      return fail(TF_ESCHEDULE, "tf_spmm_spmm: B has the shape and entry count of the inner pattern the schedule was built on, but another sparsity pattern");
    // The windowed kernel walks one staged CSR chunk for both products: B must be A.
    const bool same = (B == A) || (B->p == A->p && B->i == A->i && B->x == A->x);
    // (the kernel fetches entries four at a time and clamps the last fetch to nnz - 4: both arrays need four)
    if (s->win_wide && A->nnz >= 4 && B->nnz >= 4) {  // reads B's entries for the first product and A's for the second, in place
      TF_PHASE(s, "fused_spmm_spmm_window64_kernel", st,
               tf::launch_fused_spmm_spmm_window64(d->tiles, d->win, n_launch, B->p, B->i, B->x,
                                                   B->nnz, C->d, A->p, A->i, A->x, A->nnz, D->d, s->opts.N,
                                                   s->lds_bytes, acc, s->opts.compute_units, st));
      return TF_OK;
    }
    if (same) {
      TF_PHASE(s, "fused_spmm_spmm_window_kernel", st,
               tf::launch_fused_spmm_spmm_window(d->tiles, d->win, n_launch, d->fused_ids, A->p,
                                                 A->i, A->x, C->d, D->d, s->opts.N, s->opts.strip_cols,
                                                 s->lds_bytes, acc, st));
      return TF_OK;
    }
    if (s->lds_bytes_general > 163840)
      return fail(TF_ESCHEDULE, "tf_spmm_spmm: this schedule needs B to be the same matrix as A");
  }
  if (n_launch > 0)
    TF_PHASE(s, "fused_spmm_spmm_kernel", st,
             tf::launch_fused_spmm_spmm(d->tiles, n_launch, d->fused_ids, B->p, B->i, B->x,
                                        C->d, A->p, A->i, A->x, D->d, d->inter, s->opts.N,
                                        s->windowed ? s->lds_bytes_general : s->lds_bytes, acc, st));
  if (!s->plain_rows.empty()) {  // intermediate rows of tiles that fuse nothing
    const bool all = (int)s->plain_rows.size() == s->M;
    tf::RowsArgs a;
    a.rows = all ? nullptr : d->plain_rows;
    a.n_rows = (int)s->plain_rows.size();
    a.Ap = B->p; a.Ai = B->i; a.Ax = B->x;
    a.X = C->d; a.ldx = s->opts.N; a.x_rows = C->M; a.Y = d->inter; a.ldy = s->opts.N; a.N = s->opts.N;
    a.streaming = tf::inter_streams(s);
    tf::RowsHow how;
    how.xcd_chunk_rows = s->xcd_chunk_rows;
    TF_PHASE(s, "spmm_rows_kernel (intermediate rows)", st, tf::launch_spmm_rows(a, how, st));
  }
  return tf::run_remainder(A, s, tf::Remainder{d->inter, s->opts.N, s->opts.N, s->M, D->d, acc, 0}, false, st);
}

// What a GeMM-SpMM pass reads and writes: B (M x K), C (K x N, or N x K with c_t) and D (L x N).
struct GemmPass {
  const float *B, *C;
  int c_t, K, N;
  float *D;
  int accumulate;
  int relu_in;  // B holds a layer's output before its activation; only for schedules that relu_on_load_ok() accepts
  int relu;     // the rows of D that the row kernels write go through a ReLU
};

// One pass of a GeMM-SpMM schedule: D = A * (B * C), K and N as the schedule's kernels take them (any when nothing fuses).
static tf_status gemm_spmm_pass(const tf_csr *A, tf_schedule *s, const GemmPass &g, unsigned flags, hipStream_t st) {
  tf::DeviceSchedule *d = s->dev;
  const int n_launch = (int)s->launch_tiles.size(), ldt = tf::inter_ld(s);
  if (n_launch > 0) {
    if (s->gemm_stream)
      TF_PHASE(s, "fused_gemm_spmm_stream_kernel", st,
               tf::launch_fused_gemm_spmm_stream(d->tiles, n_launch, d->step_begin, d->step_ptr,
                                                 d->fused_rec, g.B, g.C, g.K, g.N, s->ring_rows,
                                                 A->i, A->x, g.D, d->inter, s->lds_bytes, g.accumulate, st, g.relu_in));
    else
      TF_PHASE(s, s->gemm_regw ? "fused_gemm_spmm_regw_kernel" : "fused_gemm_spmm_kernel", st,
               tf::launch_fused_gemm_spmm(d->tiles, n_launch, d->fused_ids, g.B, g.C,
                                          g.K, s->gemm_kc, A->p, A->i, A->x, g.D, d->inter,
                                          g.N, s->lds_bytes, g.accumulate, s->opts.compute_units, s->gemm_regw ? 1 : 0, st));
  }
  // Column-partitioned long rows read the most-read ("hot") intermediate rows only through their
  // hot segments.  Those rows are produced first; on request (TF_SECOND_STREAM) the hot segments
  // then run on a second stream beside the rest of the GEMM and are joined before the rows' sums.
  const bool overlap = d->side && s->plain_hot > 0 && (flags & TF_SECOND_STREAM);
  const tf::Remainder rem{d->inter, ldt, g.N, s->M, g.D, g.accumulate, g.relu};
  if (!s->plain_rows.empty()) {  // intermediate rows of tiles that fuse nothing
    const int n_plain = (int)s->plain_rows.size();
    const int placed = s->t_pos.empty() ? 0 : 1;  // the intermediate's rows stored in the order of the list
    const bool all = n_plain == s->M && s->plain_hot == 0 && !placed;
    auto gemm = [&](int first, int count) {
      const int *rows = all ? nullptr : d->plain_rows + first;
      float *Y = d->inter + (placed ? (size_t)first * ldt : 0);
      tf::GemmOut how;
      how.of_rows = n_plain;
      return tf::launch_gemm_any(g.B, g.K, g.C, g.c_t, Y, ldt, rows, !placed, count, g.K, g.N, how, s->opts.compute_units, st);
    };
    if (overlap) {
      TF_PHASE(s, "dense product (hot rows)", st, gemm(0, s->plain_hot));
      // the regrouped values (of the hot and of the cold segments) before the fork: the cold segments run on
      // this stream and are not ordered after anything the side stream does until the join
      if (tf_status rc2 = tf::ensure_segment_values(A, s, st)) return rc2;
      TF_HIP(hipEventRecord(d->fork, st));
      TF_HIP(hipStreamWaitEvent(d->side, d->fork, 0));
      if (tf_status rc2 = tf::run_hot_segments(s, rem, d->side)) return rc2;
      TF_HIP(hipEventRecord(d->join, d->side));
      if (n_plain > s->plain_hot) TF_PHASE(s, "dense product (other rows)", st, gemm(s->plain_hot, n_plain - s->plain_hot));
    } else {
      TF_PHASE(s, "dense product", st, gemm(0, n_plain));
    }
  }
  return tf::run_remainder(A, s, rem, overlap && !s->plain_rows.empty(), st);
}


// A schedule whose every intermediate row is produced by the streamed kernel straight from B (no padded copy, no
// column panels, no rows left to the row GEMM) can apply an activation to B as it is read.
static bool relu_on_load_ok(const tf_schedule *s) {
  return s->gemm_stream && !s->two_passes && s->plain_rows.empty() && s->user_K == s->opts.K && s->user_N == s->opts.N && !s->launch_tiles.empty();
}

static tf_status gemm_spmm_impl(const tf_csr *A, const tf_dense *B, const tf_dense *C, tf_dense *D,
                                tf_schedule *s, unsigned flags, void *stream, int relu_in) {
  const int c_t = (flags & TF_C_TRANSPOSED) ? 1 : 0, relu = (flags & TF_RELU) ? 1 : 0;
  tf_status rc = check_common("tf_gemm_spmm", A, C, D, s, TF_OP_GEMM_SPMM, c_t != 0);
  if (rc) return rc;
  if (!B) return fail(TF_EINVAL, "tf_gemm_spmm: B is null");
  if (B->M != A->N) return fail(TF_EINVAL, "tf_gemm_spmm: B has %d rows, A has %d columns", B->M, A->N);
  const int c_k = c_t ? C->N : C->M;
  if (B->N != s->user_K || c_k != s->user_K)
    return fail(TF_ESCHEDULE, "tf_gemm_spmm: schedule was built for K = %d, B has %d columns and C has %d rows", s->user_K, B->N, c_k);
  rc = tf::ensure_device(s);
  if (rc) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int acc = (flags & TF_ACCUMULATE) ? 1 : 0;
  tf::DeviceSchedule *d = s->dev;
  d->prof_n = 0;
  if (relu_in && !relu_on_load_ok(s)) return fail(TF_EINVAL, "tf_gemm_spmm: internal error, activation on load with a schedule that cannot apply it");
  if (s->two_passes) {
    tf_schedule *rows = s->two_passes;
    if ((rc = tf::ensure_device(rows))) return rc;
    rows->profiling = s->profiling;
    rows->dev->prof_n = 0;
    const int K = s->user_K, N = s->user_N, cus = s->opts.compute_units;
    if (s->spmm_first) {
      tf::GemmOut how;
      how.accumulate = acc;
      how.relu = relu;
      if (s->one_launch && (unsigned long long)B->M * K * 4 <= 0x80000000ull) {  // (the kernel's 32-bit offsets into B)
        tf::RowsArgs a;
        tf::RowsHow rows_how;
        if ((rc = tf::remainder_rows(A, rows, tf::Remainder{B->d, K, K, B->M, D->d, acc, relu}, st, a, rows_how))) return rc;
        a.ldy = N;
        TF_PHASE(rows, "spmm_gemm_kernel", st, tf::launch_spmm_gemm(a, rows_how, C->d, c_t, N, how, st));
        return TF_OK;
      }
      rc = tf::run_remainder(A, rows, tf::Remainder{B->d, K, K, B->M, d->inter, 0, 0, tf::inter_streams(s)}, false, st);
      if (rc) return rc;
      TF_PHASE(rows, "dense product", st, tf::launch_gemm_any(d->inter, K, C->d, c_t, D->d, N, nullptr, 0, s->L, K, N, how, cus, st));
      return TF_OK;
    }
    const int ldt = tf::inter_ld(s);
    TF_PHASE(rows, "dense product", st, tf::launch_gemm_any(B->d, K, C->d, c_t, d->inter, ldt, nullptr, 0, s->M, K, N, tf::GemmOut(), cus, st));
    return tf::run_remainder(A, rows, tf::Remainder{d->inter, ldt, N, s->M, D->d, acc, relu}, false, st);
  }
  if (tf::untiled(s)) return gemm_spmm_pass(A, s, GemmPass{B->d, C->d, c_t, s->user_K, s->user_N, D->d, acc, 0, relu}, flags, st);
  // Tiles take K in steps of 8 and N in steps of 32: zero-padded copies of B and C where the caller's differ.
  const float *Bd = B->d, *Cd = C->d;
  const bool panels = s->user_N != s->opts.N;
  if (s->user_K != s->opts.K) {
    TF_PHASE(s, "pad_kernel (B)", st, tf::launch_pad(B->d, B->M, B->N, d->Bpad, B->M, s->opts.K, st));
    Bd = d->Bpad;
  }
  if (!panels && (c_t || s->user_K != s->opts.K)) {
    if (c_t) TF_PHASE(s, "transpose_pad_kernel (C)", st, tf::launch_transpose_pad(C->d, C->M, C->N, 0, s->user_N, d->Cpad, s->opts.K, s->opts.N, st));
    else TF_PHASE(s, "pad_kernel (C)", st, tf::launch_pad(C->d, C->M, C->N, d->Cpad, s->opts.K, C->N, st));
    Cd = d->Cpad;
  }
  if (!panels) {
    rc = gemm_spmm_pass(A, s, GemmPass{Bd, Cd, 0, s->opts.K, s->opts.N, D->d, acc, relu_in, 0}, flags, st);
  } else {
    // A width the MFMA kernels do not take: one pass per column panel of opts.N columns.  The panel of C is
    // copied out (zero columns past N, zero rows past K), the pass writes a dense L x opts.N panel of D,
    // and its columns are copied (or added, with TF_ACCUMULATE) into the caller's D.
    for (int q = 0; q < s->n_panels; ++q) {
      const int c0 = q * s->opts.N, w = std::min(s->opts.N, s->user_N - c0);
      if (c_t)
        TF_PHASE(s, "transpose_pad_kernel (panel of C)", st, tf::launch_transpose_pad(C->d, C->M, C->N, c0, w, d->Cpanel, s->opts.K, s->opts.N, st));
      else
        TF_PHASE(s, "copy_cols_kernel (panel of C)", st,
                 tf::launch_copy_cols(C->d, C->M, C->N, c0, w, d->Cpanel, s->opts.K, s->opts.N, 0, s->opts.N, 0, st));
      if (tf_status rc2 = gemm_spmm_pass(A, s, GemmPass{Bd, d->Cpanel, 0, s->opts.K, s->opts.N, d->Dpanel, 0, 0, 0}, flags, st)) return rc2;
      TF_PHASE(s, "copy_cols_kernel (panel of D)", st,
               tf::launch_copy_cols(d->Dpanel, D->M, s->opts.N, 0, w, D->d, D->M, D->N, c0, w, acc, st));
    }
  }
  if (!rc && relu) TF_PHASE(s, "relu_kernel", st, tf::launch_relu(D->d, (size_t)D->M * D->N, st));
  return rc;
}

extern "C" tf_status tf_gemm_spmm(const tf_csr *A, const tf_dense *B, const tf_dense *C, tf_dense *D,
                                  tf_schedule *s, unsigned flags, void *stream) {
  return gemm_spmm_impl(A, B, C, D, s, flags, stream, 0);
}

extern "C" tf_status tf_gcn_two_layers(const tf_csr *A, const tf_dense *X, const tf_dense *W1, const tf_dense *W2, tf_dense *D,
                                       tf_schedule *s1, tf_schedule *s2, tf_dense *hidden, unsigned flags, void *stream) {
  if (!A || !X || !W1 || !W2 || !D || !s1 || !s2) return fail(TF_EINVAL, "tf_gcn_two_layers: null argument");
  if (A->M != A->N) return fail(TF_EINVAL, "tf_gcn_two_layers: A must be square (it is %d x %d)", A->M, A->N);
  const bool w_t = (flags & TF_C_TRANSPOSED) != 0;  // both weights as torch stores a layer's: outputs x inputs
  const int H = w_t ? W1->M : W1->N, w1_k = w_t ? W1->N : W1->M, w2_k = w_t ? W2->N : W2->M, w2_n = w_t ? W2->M : W2->N;
  if (w2_k != H) return fail(TF_EINVAL, "tf_gcn_two_layers: W1 has %d columns, W2 has %d rows", H, w2_k);
  if (hidden && (hidden->M != A->M || hidden->N != H))
    return fail(TF_EINVAL, "tf_gcn_two_layers: hidden is %d x %d, expected %d x %d", hidden->M, hidden->N, A->M, H);
  // every check of shape and schedule before anything is allocated or run
  if (s1->opts.op != TF_OP_GEMM_SPMM || s2->opts.op != TF_OP_GEMM_SPMM)
    return fail(TF_ESCHEDULE, "tf_gcn_two_layers: both schedules must be built for TF_OP_GEMM_SPMM");
  if (s1->L != A->M || s1->M != A->N || s2->L != A->M || s2->M != A->N)
    return fail(TF_ESCHEDULE, "tf_gcn_two_layers: the schedules were built for %d x %d and %d x %d patterns, A is %d x %d", s1->L, s1->M, s2->L, s2->M, A->M, A->N);
  if (s1->user_N != H) return fail(TF_ESCHEDULE, "tf_gcn_two_layers: the first schedule was built for N = %d, W1 has %d columns", s1->user_N, H);
  if (s2->user_K != H) return fail(TF_ESCHEDULE, "tf_gcn_two_layers: the second schedule was built for K = %d, the hidden layer has %d columns", s2->user_K, H);
  if (X->M != A->N || X->N != s1->user_K || w1_k != s1->user_K)
    return fail(TF_ESCHEDULE, "tf_gcn_two_layers: the first schedule was built for K = %d, X is %d x %d and W1 has %d rows", s1->user_K, X->M, X->N, w1_k);
  if (w2_n != s2->user_N || D->N != s2->user_N || D->M != A->M)
    return fail(TF_ESCHEDULE, "tf_gcn_two_layers: the second schedule was built for N = %d, W2 has %d columns and D is %d x %d", s2->user_N, w2_n, D->M, D->N);
  // On request (TF_FUSE_LAYERS): one launch with the hidden layer in LDS, every tile of the second schedule's two-layer
  // tiles carrying its rows through both layers (fused_gcn2_kernel).  Not the default: a tile recomputes its
  // neighbours' halo rows in both GEMMs and runs its four phases one after the other, which on the banded 262,144-row
  // pattern (K = H = N = 128) takes 0.63 ms against 0.31 ms for the two streamed launches of the composed path.
  const bool fuse_ok = !hidden && !w_t && !s2->l2_tiles.empty() && s2->user_N == s2->opts.N && s1->user_K == s1->opts.K && s1->user_K <= 256;
  if ((flags & TF_FUSE_LAYERS) && !fuse_ok)
    return fail(TF_EUNSUPPORTED, "tf_gcn_two_layers: TF_FUSE_LAYERS needs a second schedule with two-layer tiles (tf_schedule_info.two_layer_tiles: "
                "a banded pattern, widths of 32, 64 or 128), K a multiple of 8 up to 256 and no `hidden` argument");
  if (flags & TF_FUSE_LAYERS) {
    if (A->nnz != s2->nnz || (A->hash && A->hash != s2->pattern_hash))
      return fail(TF_ESCHEDULE, "tf_gcn_two_layers: the second schedule was built for another sparsity pattern than A's");
    if (tf_status rc = tf::ensure_device(s2)) return rc;
    tf::DeviceSchedule *d = s2->dev;
    d->prof_n = 0;
    hipStream_t st = static_cast<hipStream_t>(stream);
    TF_PHASE(s2, "fused_gcn2_kernel", st,
             tf::launch_fused_gcn2(d->l2_tiles, (int)s2->l2_tiles.size(), X->d, W1->d, W2->d, s1->user_K, H, s2->user_N, A->p, A->i, A->x,
                                   D->d, s2->l2_lds_bytes, (flags & TF_RELU) ? 1 : 0, (flags & TF_ACCUMULATE) ? 1 : 0, st));
    return TF_OK;
  }
  tf_dense h;
  h.M = A->M; h.N = H; h.owns = false;
  if (hidden) {
    h.d = hidden->d;
  } else {
    if (tf_status rc = tf::ensure_device(s2)) return rc;
    static std::mutex mu;  // (two threads may share a schedule object up to here; executor calls themselves are one at a time)
    std::lock_guard<std::mutex> lock(mu);
    const size_t need = (size_t)s2->L * s2->user_K;  // the hidden layer of THIS schedule: L x K
    if (!s2->dev->hidden) {
      TF_HIP(hipMalloc(reinterpret_cast<void **>(&s2->dev->hidden), need * sizeof(float)));
      s2->dev->hidden_floats = need;
    }
    if (s2->dev->hidden_floats != need)
      return fail(TF_ESCHEDULE, "tf_gcn_two_layers: the second schedule's hidden-layer buffer holds %zu floats, %zu are needed", s2->dev->hidden_floats, need);
    h.d = s2->dev->hidden;
  }
  // first layer (its schedule is checked against X and W1 there), activation, second layer.  The activation is part of
  // the first layer's row products where nothing fuses and a launch of its own over the hidden layer where tiles do --
  // unless that layer stays inside the library and the second schedule
  // streams all its rows: then the second layer's producers apply it to the hidden rows as they read them
  // (262,144-row band, K = H = N = 128: the pass over the hidden layer took 41 of the call's 343 us).
  const bool relu = (flags & TF_RELU) != 0, on_load = relu && !hidden && relu_on_load_ok(s2);
  const unsigned common = flags & (TF_SECOND_STREAM | TF_C_TRANSPOSED);
  if (tf_status rc = tf_gemm_spmm(A, X, W1, &h, s1, common | (relu && !on_load ? TF_RELU : 0u), stream)) return rc;
  return gemm_spmm_impl(A, &h, W2, D, s2, common | (flags & TF_ACCUMULATE), stream, on_load ? 1 : 0);
}

// ---- benchmark aid: per-launch times of the last executor call -------------------------

extern "C" tf_status tf_schedule_set_profiling(tf_schedule *s, int enable) {
  if (!s) return fail(TF_EINVAL, "tf_schedule_set_profiling: null argument");
  s->profiling = enable != 0;
  return TF_OK;
}

extern "C" tf_status tf_schedule_get_profile(tf_schedule *s, tf_profile *out) {
  if (!s || !out) return fail(TF_EINVAL, "tf_schedule_get_profile: null argument");
  tf_profile full;
  std::memset(&full, 0, sizeof(full));
  if (s->dev && s->profiling) {
    tf::DeviceSchedule *d = s->dev->prof_n == 0 && s->two_passes && s->two_passes->dev ? s->two_passes->dev : s->dev;
    for (int q = 0; q < d->prof_n; ++q) {
      TF_HIP(hipEventSynchronize(d->prof_ev[q][1]));
      TF_HIP(hipEventElapsedTime(&full.ms[q], d->prof_ev[q][0], d->prof_ev[q][1]));
      full.name[q] = d->prof_name[q];
    }
    full.n = d->prof_n;
  }
  return tf::emit_out("tf_schedule_get_profile", out, full, TF_SIZE_THROUGH(tf_profile, ms));
}

// ---- an executor that allocates nothing ----------------------------------------------------
//
// For callers that cannot call hipMalloc (code under HIP graph capture, serving loops, harnesses
// that forbid it): D = A*(B*C) as two row-kernel passes with the intermediate in a fixed array in
// device memory instead of a schedule's workspace.  Every GPU the library runs on holds its own
// copy of the array from the moment the library is loaded there until the process ends.

extern "C" size_t tf_noalloc_scratch_bytes(void) { return kScratchFloats * sizeof(float); }

extern "C" tf_status tf_spmm_spmm_noalloc(const tf_csr *A, const tf_csr *B, const tf_dense *C, tf_dense *D,
                                          unsigned flags, void *stream) {
  if (!A || !B || !C || !D) return fail(TF_EINVAL, "tf_spmm_spmm_noalloc: null argument");
  if (B->M != A->N) return fail(TF_EINVAL, "tf_spmm_spmm_noalloc: B has %d rows, A has %d columns", B->M, A->N);
  if (C->M != B->N) return fail(TF_EINVAL, "tf_spmm_spmm_noalloc: C has %d rows, B has %d columns", C->M, B->N);
  if (D->M != A->M || D->N != C->N)
    return fail(TF_EINVAL, "tf_spmm_spmm_noalloc: D is %d x %d, A has %d rows and C has %d columns", D->M, D->N, A->M, C->N);
  const size_t need = (size_t)B->M * C->N;
  if (need > kScratchFloats)
    return fail(TF_EUNSUPPORTED, "tf_spmm_spmm_noalloc: the intermediate (%d x %d floats, %zu bytes) exceeds the fixed scratch of %zu bytes; "
                "use tf_spmm_spmm, whose schedule allocates its workspace", B->M, C->N, need * sizeof(float), kScratchFloats * sizeof(float));
  float *T = nullptr;
  if (tf_status rc = scratch_of_current_device(&T)) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  // every intermediate row is overwritten (rows without entries with zeros), so nothing of the
  // previous call's contents is read
  tf::RowsArgs first = all_rows(B, C->d, T, C->N), second = all_rows(A, T, D->d, C->N);
  second.streaming = 1;
  second.accumulate = (flags & TF_ACCUMULATE) ? 1 : 0;
  TF_HIP(tf::launch_spmm_rows(first, tf::RowsHow(), st));
  TF_HIP(tf::launch_spmm_rows(second, tf::RowsHow(), st));
  return TF_OK;
}

extern "C" tf_status tf_spmm(const tf_csr *A, const tf_dense *X, tf_dense *Y, unsigned flags, void *stream) {
  if (!A || !X || !Y) return fail(TF_EINVAL, "tf_spmm: null argument");
  if (X->M != A->N || Y->M != A->M || X->N != Y->N)
    return fail(TF_EINVAL, "tf_spmm: shapes A %d x %d, X %d x %d, Y %d x %d", A->M, A->N, X->M, X->N, Y->M, Y->N);
  tf::RowsArgs a = all_rows(A, X->d, Y->d, X->N);
  a.streaming = 1;
  a.accumulate = (flags & TF_ACCUMULATE) ? 1 : 0;
  TF_HIP(tf::launch_spmm_rows(a, tf::RowsHow(), static_cast<hipStream_t>(stream)));
  return TF_OK;
}

extern "C" tf_status tf_spmm_scheduled(const tf_csr *A, const tf_dense *X, tf_dense *Y, tf_schedule *s, unsigned flags, void *stream) {
  if (!A || !X || !Y || !s) return fail(TF_EINVAL, "tf_spmm_scheduled: null argument");
  if (!s->rows_only) return fail(TF_ESCHEDULE, "tf_spmm_scheduled: the schedule is not one of tf_inspect_spmm");
  if (tf_status rc = check_pattern("tf_spmm_scheduled", A, s)) return rc;
  if (X->M != A->N || Y->M != A->M || X->N != Y->N || X->N > s->user_N)
    return fail(TF_EINVAL, "tf_spmm_scheduled: shapes A %d x %d, X %d x %d, Y %d x %d, schedule for N up to %d", A->M, A->N, X->M, X->N, Y->M, Y->N, s->user_N);
  if (tf_status rc = tf::ensure_device(s)) return rc;
  s->dev->prof_n = 0;
  return tf::run_remainder(A, s, tf::Remainder{X->d, X->N, X->N, X->M, Y->d, (flags & TF_ACCUMULATE) ? 1 : 0, (flags & TF_RELU) ? 1 : 0}, false,
                           static_cast<hipStream_t>(stream));
}

extern "C" tf_status tf_gemm(const tf_dense *X, const tf_dense *W, tf_dense *Y, void *stream) {
  return tf_gemm_ex(X, W, Y, nullptr, 0, stream);
}

extern "C" tf_status tf_gemm_ex(const tf_dense *X, const tf_dense *W, tf_dense *Y, const tf_dense *mask, unsigned flags, void *stream) {
  if (!X || !W || !Y) return fail(TF_EINVAL, "tf_gemm: null argument");
  const bool w_t = (flags & TF_C_TRANSPOSED) != 0;
  const int K = X->N, N = Y->N, M = X->M;
  if ((w_t ? W->N : W->M) != K || (w_t ? W->M : W->N) != N || Y->M != M)
    return fail(TF_EINVAL, "tf_gemm: shapes X %d x %d, W %d x %d%s, Y %d x %d", X->M, X->N, W->M, W->N, w_t ? " (transposed)" : "", Y->M, Y->N);
  if (mask && (mask->M != M || mask->N != N)) return fail(TF_EINVAL, "tf_gemm: mask is %d x %d, Y is %d x %d", mask->M, mask->N, M, N);
  hipStream_t st = static_cast<hipStream_t>(stream);
  tf::GemmOut how;
  how.mask = mask ? mask->d : nullptr;
  TF_HIP(tf::launch_gemm_any(X->d, K, W->d, w_t ? 1 : 0, Y->d, N, nullptr, 0, M, K, N, how, tf::default_compute_units(), st));
  return TF_OK;
}

extern "C" size_t tf_weight_grad_workspace(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  return tf::plan_weight_grad(M, N, K, tf::default_compute_units()).partial_floats() * sizeof(float);
}

static tf_status weight_grad_task(const char *who, const tf_dense *G, const tf_dense *X, tf_dense *Y, float *workspace, tf::WeightGradTask *t) {
  if (!G || !X || !Y) return fail(TF_EINVAL, "%s: null argument", who);
  if (G->M != X->M || Y->M != G->N || Y->N != X->N)
    return fail(TF_EINVAL, "%s: shapes G %d x %d, X %d x %d, Y %d x %d", who, G->M, G->N, X->M, X->N, Y->M, Y->N);
  *t = tf::plan_weight_grad(G->M, G->N, X->N, tf::default_compute_units());
  if (t->partial_floats() && !workspace) return fail(TF_EINVAL, "%s: %zu bytes of workspace needed", who, t->partial_floats() * sizeof(float));
  t->G = G->d;
  t->X = X->d;
  t->Y = Y->d;
  t->partial = workspace;
  return TF_OK;
}

extern "C" tf_status tf_weight_grad(const tf_dense *G, const tf_dense *X, tf_dense *Y, float *workspace, void *stream) {
  tf::WeightGradTask t;
  if (tf_status rc = weight_grad_task("tf_weight_grad", G, X, Y, workspace, &t)) return rc;
  TF_HIP(tf::launch_weight_grads(t, nullptr, static_cast<hipStream_t>(stream)));
  return TF_OK;
}

extern "C" tf_status tf_weight_grad_pair(const tf_dense *G1, const tf_dense *X1, tf_dense *Y1, float *workspace1, const tf_dense *G2, const tf_dense *X2,
                                         tf_dense *Y2, float *workspace2, void *stream) {
  tf::WeightGradTask a, b;
  if (tf_status rc = weight_grad_task("tf_weight_grad_pair", G1, X1, Y1, workspace1, &a)) return rc;
  if (tf_status rc = weight_grad_task("tf_weight_grad_pair", G2, X2, Y2, workspace2, &b)) return rc;
  TF_HIP(tf::launch_weight_grads(a, &b, static_cast<hipStream_t>(stream)));
  return TF_OK;
}
