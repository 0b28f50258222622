// Internal declarations shared by the host-side inspector, the C ABI and the HIP
// kernels of libtilefusion_hip.  Not installed; the public surface is
// include/tilefusion_hip.h.
#pragma once
#include <cstdarg>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "tilefusion_hip.h"

namespace tf {

constexpr int kMaxLds = 163840;  // LDS per workgroup on gfx950
// Streamed GeMM-SpMM runs: two buffers of 64 x 32 values of B, each as three bf16 parts.
constexpr int kStreamStageBytes = 24576;
// ... and a row's entries, as many slots as a group of `lanes` lanes (8, 16 or 32) has.  Lane l reads four slots from base + 4 stream_quarter(l): of each
// sixteen entries its quad's lanes hold a quarter each, of a group's eight two lanes the same half.
constexpr int stream_quarter(int l, int lanes) { return l & 3 & (lanes / 4 - 1); }

// One fused tile = one workgroup.  The workgroup computes intermediate rows
// [prod_begin, prod_end) into LDS, stores rows [wb_begin, wb_end) of them to the
// intermediate in HBM (the ones remainder rows will read), then computes the
// second-op rows ids[cons_begin .. cons_end) out of LDS.
struct TileDesc {
  int prod_begin, prod_end;
  int own_begin, own_end;
  int wb_begin, wb_end;
  int cons_begin, cons_end;
};
static_assert(sizeof(TileDesc) == 32, "TileDesc is read as two int4 by the kernels");

// A chunk of one long remainder row: stored entries [k_begin, k_end) of `row`,
// reduced by a whole workgroup into partial[slot].
struct LongChunk {
  int row, k_begin, k_end, slot;
};
// All partials of one long row: D[row] = sum partial[first .. first+count).
struct LongRow {
  int row, first, count, pad;
};

// A tile that carries its rows through two GCN layers (tf_gcn_two_layers): it owns the rows [o0, o1) of D, which
// read the rows [h0, h1) of the hidden layer, which read the rows [t0, t1) of the first layer's intermediate.
struct Tile2 {
  int o0, o1, h0, h1, t0, t1;
  int b_off;  // floats of LDS in front of the tile's slab B (its slab A: the first intermediate, then the second)
  int c_off;  // ... and in front of its copy of A's rows [min(o0, h0), max(o1, h1)): row pointers, columns, values
};
static_assert(sizeof(Tile2) == 32, "Tile2 is read as two int4 by the kernel");
constexpr int kTile2Pad = 4;                 // floats behind every slab row (tf_gcn2.hip: kG2Pad)
constexpr int kTile2StageFloats = 2 * 64 * 36;  // the two staging buffers of X (tf_gcn2.hip: kG2StageFloats)

// Operands of the row kernel (tf_rows.hip).  Y[i,:] (+)= sum over row r's entries of Ax[k] * X[Ai[k],:], i = rows[q] (q without
// a list), r = q with `compact`, else i.
struct RowsArgs {
  const int *rows = nullptr;
  int n_rows = 0;
  const int *Ap = nullptr, *Ai = nullptr;
  const float *Ax = nullptr, *X = nullptr;
  const int *val_first = nullptr;  // with `compact`: where row q's values start in Ax (null: at Ap[q], as its columns in Ai)
  int ldx = 0;
  unsigned x_rows = 0;  // rows of X
  float *Y = nullptr;
  int ldy = 0, N = 0;
  int accumulate = 0, streaming = 0, compact = 0, relu = 0;
  // rows of Y without entries that are not among n_rows: cleared on the way (n_zero > 0 needs n_rows > 0)
  const int *zero_rows = nullptr;
  int n_zero = 0;
  // chunks of long rows, a workgroup each; slot < 0: the row's only chunk, which goes straight to Y
  // (their k_begin and k_end count in chunk_Ai and chunk_Ax, the matrix' own arrays)
  const LongChunk *chunks = nullptr;
  unsigned n_chunks = 0;
  const int *chunk_Ai = nullptr;
  const float *chunk_Ax = nullptr;
  float *partial = nullptr;
  // rows of several chunks: which of long_rows a chunk belongs to (-1: its row has no other), and how many of each have arrived
  const int *chunk_long = nullptr;
  const LongRow *long_rows = nullptr;
  unsigned *arrived = nullptr;
  unsigned chunk_blocks = 0;          // set by the launcher
  int n_blocks = 0, per_xcd = 0, slices = 1;  // set by the launcher
  int sweep_steps = 0;                        // ... for sweep_rows_kernel: steps in which its window passes over X,
  unsigned sweep_bytes = 0;                   // and by how much in each
};
struct RowsHow {
  int xcd_chunk_rows = 0;   // how row blocks are dealt to the XCDs (tf_inspect_opts.xcd_chunk_rows)
  long long spread_entries = 0;  // of all rows where their columns are spread over X alike, rising in each row (0: they are not, or nobody knows)
  int flagged = 0;          // columns carry the "cold" mark
};

// What becomes of a dense product's values on their way to Y (tf_dense.hip).
struct GemmOut {
  const float *mask = nullptr;  // of Y's shape: 0 where it is zero or less (the derivative of a ReLU whose output it is)
  int accumulate = 0;           // Y += the product
  int relu = 0;
  int of_rows = 0;              // rows of the whole product where it comes in parts: all are computed by the same kernel (0: its own)
};

// Y = G^T X, G M x N and X M x K, and how launch_weight_grads cuts it (tf_dense.hip).
struct WeightGradTask {
  const float *G = nullptr, *X = nullptr;
  float *Y = nullptr, *partial = nullptr;
  int M = 0, N = 0, K = 0;
  int few = 0;  // in one launch, without a workspace; of the cuts below only k_chunks is set
  int nb = 0, kb = 0, n_chunks = 0, k_chunks = 0, groups = 0, waves = 0;  // waves: of a workgroup
  int blocks() const { return few ? n_chunks * k_chunks : groups * n_chunks * k_chunks; }  // workgroups
  size_t partial_floats() const { return few ? 0 : (size_t)blocks() * nb * kb * 256; }
};

// Runs over the 27-point stencil (tf_box.hip): columns of 2 q x by points.  LDS holds two planes of C with two points around the
// column and two of the intermediate with one.
constexpr int kBoxBlock = 1024, kBoxMaxY = 6;
constexpr int box_lds(int q, int by) { return 512 * ((2 * q + 4) * (by + 4) + (2 * q + 2) * (by + 2)) + 16 * 108 * (2 * q + 1); }
// Runs over the 7-point stencil (tf_star.hip): columns of 16 by up to 8 points, 32 columns of C wide.  LDS holds two planes of C with two points around
// the column and two of the intermediate in the same places, lines of 20 points of 128 bytes, and a line that what nobody wants is read from.
constexpr int kStarX = 16, kStarMaxY = 8, kStarLine = (kStarX + 4) * 128, kStarBlock = 768;
constexpr int star_lds(int by) { return kStarLine * (2 * ((by + 4) + (by + 2)) + 1); }
// ... and over the 5-point stencil of a 2D grid, which is its one with a line for a plane: columns of up to 94 points of a line.
constexpr int kFlatX = 94, kFlatBlock = (kFlatX + 2) / 2 * 8, kFlatLine = (kFlatX + 6) * 128, kFlatRuns = 2;  // runs a compute unit holds
constexpr int flat_lds() { return kFlatLine * 4; }
// What either kernel of such runs is launched with.
struct BoxArgs {
  int star = 0;  // the 7-point (ny = 1: 5-point) stencil instead of the 27-point one
  int nx = 0, ny = 0, nz = 0, N = 0;
  int q = 0, bx = 0, by = 0, tx = 0, ty = 0, zlen = 0, strips = 0, n_runs = 0;  // columns in x (bx points) and y, planes a run, strips of 64 columns (star: 32)
  int per_xcd = 0, streaming = 1;                                // set by the launcher
  unsigned val_bytes = 0;                                        // of Ax and of Bx
  const float *Ax = nullptr, *Bx = nullptr, *C = nullptr;
  float *D = nullptr;
};

struct DeviceSchedule;  // device copies + workspace, defined in tf_api.cpp

// Marching runs: LDS layout and list format shared by the inspector, the validator and the kernel.
constexpr int kMarchW = 8;               // entries per ELL row when no row of either pattern has more: a lane of a quad holds two
constexpr int kMarchWideW = 32;          // ... and when one has (up to 32: longer rows do not march): a lane of a group holds two
// entries per ELL row in a schedule whose longest row has `width` entries
constexpr int march_ell_stride(int width) { return width <= kMarchW ? kMarchW : kMarchWideW; }
constexpr int kMarchRowBytes = 256;      // an LDS slot: 64 columns of one row
constexpr int kMarchTabBytes = 4096;     // per-iteration table of a run, staged at the start of LDS
constexpr int kMarchMaxIter = kMarchTabBytes / 16 - 2;  // (16 bytes of table per iteration)
constexpr int kMarchZeroOff = kMarchTabBytes;                    // a row of zeros, read by padding entries
constexpr int kMarchTrashOff = kMarchTabBytes + kMarchRowBytes;  // a row that takes what lane groups without work write
constexpr int kMarchSlot0 = kMarchTabBytes + 2 * kMarchRowBytes; // first slot
constexpr int kMarchSrcA = 1 << 30;      // flag in march_ell_src: the value is one of A's (else of B's)
constexpr int kMarchGroups = 32;         // lane groups (of 16 lanes) per workgroup
// rows one lane group takes per iteration, at most (the kernel's register sets): intermediate rows,
// second-op rows, rows of C
constexpr int kMarchTpg = 3, kMarchDpg = 2, kMarchLpg = 5;

}  // namespace tf

struct tf_schedule {
  tf_inspect_opts opts{};  // resolved (no zero "default" fields left)
  int L = 0, M = 0;
  int lds_bytes = 0;          // dynamic LDS of the fused kernel: intermediate slab (+ GEMM staging)
  int lds_bytes_general = 0;  // the same for the kernel that gathers C from HBM (fallback of windowed tiles)
  bool windowed = false;      // tiles stage their window of C in LDS (win holds the windows)
  bool win_wide = false;      // ... in 64-column strips on the 1024-thread kernel (entries read in place)
  long long inner_nnz = 0;    // stored entries of the inner pattern the windows were built from
  std::vector<int> win;       // [2*n_tiles] first,last+1 row of C read by the tile's producer rows
  int slab_rows = 0;          // max producer rows of any tile
  int user_K = 0;             // K as given; opts.K is K rounded up to a multiple of 8 (what the kernels see)
  int user_N = 0;             // N as given; GeMM-SpMM with a width the MFMA kernels do not take (N % 32, N > 256) runs
  int n_panels = 1;           // as n_panels column panels of opts.N columns each, the last one zero-padded
  // Where it is faster than the tiles (see choose_two_passes in tf_inspector.cpp) the executor runs two products through an
  // intermediate in HBM, A's by this schedule of tf_inspect_spmm.  spmm_first (GeMM-SpMM): as (A B) C.
  tf_schedule *two_passes = nullptr;
  bool spmm_first = false;
  bool one_launch = false;    // ... in one kernel that multiplies the rows of A B by C in LDS (spmm_gemm_kernel)
  bool rows_only = false;     // a schedule of tf_inspect_spmm: one product, every row in the remainder lists
  int gemm_kc = 0;            // rows of C staged in LDS per step (GeMM-SpMM)
  bool gemm_regw = false;     // GeMM-SpMM tiles keep C in registers (no staging; slab rows padded)
  int slab_ld = 0;            // floats between two slab rows of the general / GeMM-SpMM tile kernels
  bool gemm_stream = false;   // GeMM-SpMM tiles are long runs streamed through a ring of ring_rows slab rows
  int ring_rows = 0;
  int stream_step_cap = 0;    // rows a step of a streamed run may hold (all but the last step)
  int stream_max_len = 0;     // entries a fused row of a streamed run may have
  std::vector<int> tile_step;    // per tile: first entry of its steps in step_ptr (-1: fuses nothing)
  std::vector<int> launch_step;  // the same for launch_tiles
  std::vector<int> step_ptr;     // per streamed tile steps+2 offsets into fused_ids: rows of step q are
                                 // [step_ptr[q], step_ptr[q+1]), computed while rows 64q.. are produced
  std::vector<int> view_step_ptr;  // step_ptr with offsets counted from each tile's first fused id
  std::vector<int> fused_rec;    // (row, first entry, end, 0) per fused id of a streamed schedule
  std::vector<tf::TileDesc> tiles;
  std::vector<tf::TileDesc> launch_tiles;  // the tiles that fuse something: one workgroup each
  std::vector<int> plain_rows;      // intermediate rows of tiles that fuse nothing, computed by the
                                    // row kernels -- only the rows some remainder row reads
  int plain_hot = 0;                // with long_part: the first plain_hot of them are the rows of the hot
                                    // partitions (produced first, so that the hot segments can start early)
  bool profiling = false;           // executors record events around every launch
  std::vector<int> fused_ids;       // second-op rows per tile, tile after tile
  std::vector<int> rem_rows;        // remainder rows handled one row per lane group, ordered by
                                    // length class so that a workgroup's rows cost about the same
  bool rem_identity = false;        // rem_rows is 0..L-1 in order
  bool rem_sweep = false;           // ... whose columns are spread over all alike (RowsHow::spread_entries)
  int reads_even = -1;              // no column of A is read much more often than the others (-1: not counted)
  std::vector<int> zero_rows;       // second-op rows without entries, when many: their rows of D are cleared by a
                                    // fill kernel instead of taking a lane group each in the row kernel
  // When the list is not the identity, its rows are also kept as a CSR of their own in list order
  // (row q of it is row rem_rows[q] of A): rem_ptr [n + 1], rem_col, and rem_src = where each entry
  // sits in A's arrays (the executor copies the values from there).
  std::vector<int> rem_ptr, rem_col, rem_src;
  bool rem_flagged = false;  // rem_col carries the "cold" mark in the top bit of some columns (short_row_hot_bytes)
  int rem_hot_rows = 0;      // intermediate rows left unmarked
  int xcd_chunk_rows = 0;           // rows per XCD turn of the row kernels (0: one contiguous run per XCD)
  int row_deal = 0;  // how the row kernels deal their rows to the XCDs: xcd_chunk_rows where given, else the inspector's choice
  std::vector<tf::LongChunk> long_chunks;
  std::vector<tf::LongRow> long_rows;
  // Long rows cut by column instead (long_part): the most-read intermediate rows are dealt to 8
  // partitions, one per XCD, small enough to stay in that XCD's L2; a long row's entries are
  // regrouped into segments of one partition (or of none: "cold") and of at most 64 entries,
  // each worked on like a short row by the XCD that caches its partition.  long_rows then holds
  // first/count into lrow_seg.
  bool long_part = false;
  int seg_per_xcd = 0;            // hot segments per partition, padded with empty ones
  int hot_cols = 0;               // intermediate rows in the 8 partitions together
  std::vector<int> seg_ptr;       // [n_seg + 1] into seg_src/seg_col: partition 0's segments, 1's, ..., 7's, the cold ones
  std::vector<int> seg_src;       // per regrouped entry: its index in A's arrays
  std::vector<int> seg_col;       // per regrouped entry: its column
  std::vector<int> lrow_seg;      // per long row (first, count of tf::LongRow): the partial-sum slots it adds up, in order:
                                  // segments, or for a row of more than 32 segments groups of up to 32 of them
  std::vector<tf::LongRow> seg_groups;  // such groups: row = the group's slot (n_seg + its index), first/count into lrow_seg
  // Marching runs (SpMM-SpMM on stencil-like patterns whose dependences no contiguous tile holds): a run
  // is one workgroup that walks a sequence of steps (a column of grid points, plane by plane) and keeps
  // the rows of C and of the intermediate that its next rows need in numbered LDS slots of one
  // 64-column row each.  Iteration i of a run has the C rows of load list i in LDS, computes the ELL rows
  // [row_ptr[2i], row_ptr[2i+1]) -- the intermediate rows first needed by the run's step i, into slots
  // (halo rows of neighbouring runs are recomputed) -- and, after a barrier, the ELL rows
  // [row_ptr[2i+1], row_ptr[2i+2]) -- the second-op rows of step i, to D -- while the C rows of list i+1
  // go to their slots.  Every entry of an ELL row names the LDS byte offset of the row it reads; the
  // inspector assigns the slots so that a row stays until its last reader has run.
  bool march = false;
  // GeMM-SpMM schedules in which nothing fuses and every gather goes through the schedule's own copies of the columns:
  // t_pos[c] = where row c of the intermediate is stored (its place in plain_rows: the rows of the hot partitions
  // first, the others by falling number of reads), -1 for rows nobody reads.  Empty: rows at their own index.
  std::vector<int> t_pos;
  int march_declined = TF_MARCH_NOT_TRIED;  // why there are no marching runs (TF_MARCH_*), TF_MARCH_BUILT when there are
  int march_grid[3] = {0, 0, 0};     // the grid the runs were cut from (x fastest)
  int march_tile[2] = {0, 0};        // grid points per run and plane: x, y
  int march_slots = 0;               // LDS slots in use by the fullest run
  int march_width = tf::kMarchW;         // entries of the longest row of either pattern (the kernel takes only that many pairs of a row, five at least)
  int march_tpg = 0, march_dpg = 0, march_lpg = 0;  // intermediate rows / second-op rows / C rows a lane group handles per iteration, at most
  std::vector<int> march_runs;       // (first iteration, iterations) per run
  std::vector<int> march_row_ptr;    // [2 * iterations + 1] into the ELL rows
  std::vector<int> march_load_ptr;   // [iterations + 1] into the load list
  std::vector<int> march_load;       // (row of C, LDS byte offset) pairs
  std::vector<int> march_row_out;    // per ELL row: >= 0 row of D, < 0 ~(LDS byte offset) of an intermediate row
  std::vector<int> march_row_id;     // per ELL row: the matrix row it computes (of B when out < 0, of A otherwise)
  std::vector<int> march_ell_off;    // [march_ell_stride(march_width) per ELL row] LDS byte offset of the row read (the zero row for padding)
  std::vector<int> march_ell_src;    // ... and where its value comes from: index into B's values, or into A's
                                     // with kMarchSrcA set; -1 for padding (value 0)
  // Runs over a grid whose 27-, 7- or 5-point stencil both patterns are: marching runs of a kernel of their own, without any of the lists above.
  bool box = false;
  bool box_beside = false;  // ... that stand in for two products: the schedule is as good for A's pattern alone, with any inner matrix
  bool box_room = false;    // ... or stand where the runs of lists would be two products: with room for an intermediate, for calls they are not for
  tf::BoxArgs box_runs;
  double box_us = 0, box_other_us = 0;  // what they are expected to take, and two products
  // Two-layer tiles (GeMM-SpMM schedules of a square matrix with K and N of 32, 64 or 128, when every tile's two
  // halos fit LDS): what tf_gcn_two_layers runs when this is the second layer's schedule.  l2_lds_bytes: the LDS
  // of the fullest tile (slab A in front, slab B -- X staging, then the hidden rows -- behind it).
  std::vector<tf::Tile2> l2_tiles;
  int l2_lds_bytes = 0;
  long long fused_nnz = 0;
  int n_writeback_rows = 0;
  long long n_producer_rows = 0;
  // MultiDimensionalSet-layout view
  std::vector<int> ptr1, ptr2, ker_begin, id, type, tile_range, writeback;
  // pattern fingerprint, checked by the executors against their operands
  long long nnz = 0;
  uint64_t pattern_hash = 0;  // tf_pattern_hash of the pattern the schedule was built from
  uint64_t inner_hash = 0;    // ... and of the inner pattern, when one was given (0: none)
  tf::DeviceSchedule *dev = nullptr;
};

namespace tf {

tf_status fail(tf_status code, const char *fmt, ...);

// Out-structs (tf_device_info, tf_schedule_info, tf_schedule_view, tf_profile) begin with the size the
// caller was compiled with.  `full` is the struct as this library knows it; the caller gets its first
// min(struct_size, sizeof(T)) bytes and keeps its own struct_size, so nothing is written behind a
// struct that is shorter than this library's.  min_size = the struct's size in its first version.
template <class T> tf_status emit_out(const char *who, T *out, T &full, size_t min_size) {
  const size_t have = out->struct_size;
  if (have < min_size)
    return fail(TF_EINVAL, "%s: struct_size is %zu, the struct's first version has %zu bytes (set struct_size to sizeof of the struct before the call)",
                who, have, min_size);
  full.struct_size = have;
  std::memcpy(static_cast<void *>(out), &full, have < sizeof(T) ? have : sizeof(T));
  return TF_OK;
}
// size of struct T up to and including its member m
#define TF_SIZE_THROUGH(T, m) (offsetof(T, m) + sizeof(((T *)nullptr)->m))
// tf_march.cpp: builds marching runs into S (returns false, S untouched, when the pattern does not
// suit them), and checks such a schedule exactly against both patterns.
bool build_march(tf_schedule *S, int M, const int *Ap, const int *Ai, const int *Bp, const int *Bi,
                 const tf_inspect_opts &o, const tf_inspect_opts &given);
tf_status validate_march(const tf_schedule *s, int M, const int *Ap, const int *Ai, const int *Bp, const int *Bi);
// The same for runs over a 27-point stencil.
bool build_box(tf_schedule *S, int M, const int *Ap, const int *Ai, const int *Bp, const int *Bi,
               const tf_inspect_opts &o, const tf_inspect_opts &given);
tf_status validate_box(const tf_schedule *s, int M, const int *Ap, const int *Ai, const int *Bp, const int *Bi);
bool asks_for_tiles(const tf_inspect_opts &given);
bool march_as_two_products(const tf_schedule *S);
int rows_in_order_deal(int L, int M, int N, const int *Ap);
void release_device_schedule(DeviceSchedule *d);
int default_compute_units();

}  // namespace tf
