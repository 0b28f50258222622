// How the row kernels (tf_rows.hip) deal a row's columns to lanes and XCDs.  Host rules without a HIP header, so that a
// test can enumerate which lane stores which column.
#pragma once
#include <algorithm>
#include <climits>

#include "tf_internal.h"

namespace tf {

// What one lane stores of a row of N columns: its V columns, or the last V when they reach past the end (two
// lanes of a group then store some of the same values).
template <int V> constexpr int clamp_col(int c, int N) { return c < N - V ? c : N - V; }

// Lanes a row of N columns takes: V = 4 columns each (any N of four or more: a lane whose columns would reach past the
// row's end takes the last four), one each for narrower rows.  With accumulation into a row longer than the 256 columns of
// one pass, a last lane of a later pass must not fall back into columns the pass before has added to.
struct RowShape { int V, LPR; };
inline RowShape row_shape(int N, int accumulate) {
  const int V = N < 4 || (accumulate && N > 256 && N % 4 != 0) ? 1 : 4;
  int LPR = V == 1 ? (N < 4 ? 4 : 64) : 2;
  if (V == 4)
    while (LPR * 4 < N && LPR < 64) LPR *= 2;
  return {V, LPR};
}

// Slices of 32 columns, a cache line each, where a slice is a few times an XCD's L2 and X is not: gathers that came out of
// the Infinity Cache then hit.  One product of an Erdos-Renyi graph (10 - 12 entries a row), whole rows / slices: N = 128,
// 10,000 rows 6.4 / 6.4 us, 20,000 14.5 / 10.1, 50,000 46 / 34, 100,000 83 / 75, 200,000 170 / 171; N = 64, 50,000 rows 21 / 19,
// 100,000 41 / 39, and not on stencils (16 / 16.5).  Rows that do not start at a line would share lines between slices
// (N = 100, 50,000 rows: 41 / 65); values read in place cost a line a row and slice, more than two slices gain (N = 64, 100,000 rows:
// 41.8 / 42.7).
// The last slice's last lane may not reach back into the slice before it where Y is added to: workgroups of two XCDs would both
// add to those columns, and one that loads after the other has stored adds twice.  (N = 97 .. 99: whole rows.)
// A few long rows' chunks beside them, which take all columns slice by slice, do not matter, many do (Erdos-Renyi with some rows of more than 32
// entries, N = 128, whole rows / slices, two products: 20,000 rows 38.9 / 29.0, 28,334 rows of 16 56.8 / 40.0, 50,000 rows of 17 118 / 88; N = 64, 60,000 rows
// 65.8 / 58.1; a layer forward and backward, 100 -> 128, 60,000 rows 216 / 194; power-law graphs, a tenth of whose rows are long: 2^14 nodes, 96 -> 128 34 / 36,
// 2^16 50 / 54).
constexpr int kSliceCols = 32;
inline int slices_for(const RowsArgs &a) {
  if (a.ldx % 32 != 0 || (reinterpret_cast<uintptr_t>(a.X) & 127u) || (long long)a.n_chunks * 256 > a.n_rows) return 1;
  const long long bytes = (long long)a.x_rows * a.ldx * 4;
  int slices = 1;
  if (a.N > 96 && a.N <= 128 && a.x_rows >= 16000 && bytes <= (64LL << 20)) slices = 4;
  else if (a.N > 48 && a.N <= 64 && a.compact && !a.val_first && a.x_rows >= 24000 && bytes <= (40LL << 20)) slices = 2;
  if (a.accumulate && a.N - 4 < (slices - 1) * kSliceCols) slices = 1;
  return slices;
}

// sweep_rows_kernel: rows of some entries each, spread over an X that no L2 holds and the Infinity Cache does.  Erdos-Renyi graphs, one product,
// the other kernel / this one (us; a layer's two products with values read in place in brackets): N = 64, 60,000 rows of 11 20.3 / 20.8
// (47.2 / 41.8), 100,000 38.2 / 34.1 (83 / 69), 200,000 82.9 / 77.7 (177 / 156); N = 128, 60,000 38.5 / 38.4 (88 / 77),
// 100,000 77.5 / 67.0 (173 / 137), 200,000 168 / 156 (344 / 315), 400,000 335 / 334 (690 / 656); N = 32, 200,000 rows 42.4 / 40.4 (95 / 83); N = 16,
// 250,000 rows 44.1 / 36.9 (106 / 78).  Not below 15 MB of X (36,000 rows of 13, N = 100: 21.3 / 23.2), where it outgrows the Infinity Cache (10^6 rows of
// 9, N = 64: 355 / 359), for fewer than 5.5 entries a row (200,000 rows of 4, N = 64: 35.8 / 37.2), or where a row is three quarters of a lane group
// (120,000 rows, N = 80: 68 / 70).  Four slices of whole lines of 128 columns hold out longer, up to 20 MB (two products, kept values, rows of 6 / 9 / 11 / 17:
// 30,000 rows 24.2 / 28.5 / 31.8 / 43.4 against 27.6 / 33.8 / 37.3 / 53.2, 34,000 26.8 / 32.4 / 36.4 / 50.3 against 29.8 / 34.6 / 39.4 / 56.2, 38,000 30.0 / 36.9 / 41.6 /
// 57.9 against 32.2 / 37.9 / 41.6 / 59.7, 42,000 33.5 / 42.0 / 47.5 / 67.7 against 35.5 / 42.9 / 49.1 / 70.8, 46,000 37.3 / 47.2 / 54.2 / 76.5 against 37.9 / 45.9 / 50.6 / 71.1; a layer
// of 64 -> 128, values read in place, rows of 17: 30,000 rows 77.3 against 79.3, 34,000 89.9 against 89.0, 42,000 106 against 103.5).
constexpr int kSweepRows = 4, kSweepEntries = 16;
constexpr bool sweep_fits(long long x_rows, int N, long long rows, long long entries) {
  return N >= 4 && (N <= 64 || (N > 96 && N <= 128)) && x_rows * N * 4 >= (N == 128 ? 20000000 : 15000000) && x_rows * N * 4 <= (256ll << 20) && 2 * entries >= 11 * rows;
}
// Lanes a row takes, column slices, and the steps in which the limit passes over X.  Slices as above where rows start at a line, of 64 columns where four
// of 32 do not pay: as long as an XCD's slice is small enough that most of it is read by more than one row in flight (N = 128, whole rows / two slices / four:
// 60,000 rows 45 / 38.4 / 38.8, 100,000 78 / 69.5 / 67, 200,000 162 / 156 / 164; N = 64, whole / two, 100,000 36.5 / 34.1, 200,000 79.5 / 77.7,
// 400,000 168 / 185).  More steps than entries, or rows that have two close together fall behind (steps per entry 1 / 1.5 / 2: N = 64, 60,000 rows
// 20.2 / 20.8 / 22.6, 100,000 35.6 / 34.1 / 36.6, 200,000 85 / 80 / 78).
struct SweepShape { int LPR = 0, slices = 1, steps = 0; };
inline SweepShape sweep_for(const RowsArgs &a, const RowsHow &how) {
  SweepShape s;
  const long long bytes = (long long)a.x_rows * a.ldx * 4;
  if (row_shape(a.N, a.accumulate).V != 4 || how.spread_entries <= 0 || how.flagged || how.xcd_chunk_rows != 0 || a.n_chunks > 0 || a.rows || a.n_zero > 0 ||
      !sweep_fits(a.x_rows, a.N, a.n_rows, how.spread_entries) || bytes > 0x80000000ll)
    return s;
  s.LPR = a.N <= 16 ? 4 : row_shape(a.N, 0).LPR;
  if (a.ldx % 32 == 0 && !(reinterpret_cast<uintptr_t>(a.X) & 127u)) {
    if (a.N > 96 && bytes > (40 << 20) && bytes <= (64 << 20)) s.LPR = 8, s.slices = 4;
    else if (a.N > 96) s.LPR = 16, s.slices = 2;
    else if (a.N > 48 && bytes <= (64 << 20)) s.LPR = 8, s.slices = 2;
    // (as in slices_for)
    if (a.accumulate && a.N - 4 < (s.slices - 1) * s.LPR * 4) s.LPR = row_shape(a.N, 0).LPR, s.slices = 1;
  }
  s.steps = (int)((bytes > (32 << 20) ? 4 : 3) * how.spread_entries / (2 * a.n_rows)) + 1;
  return s;
}

// spmm_gemm_kernel: rows of A X a workgroup holds in LDS, and the LDS they take (K columns in steps of 16, four floats behind
// each row).
constexpr int spmm_gemm_rows(int n_rows) { return n_rows < 24000 ? 16 : 64; }
constexpr long long spmm_gemm_lds(int n_rows, int K) { return spmm_gemm_rows(n_rows) * (((long long)K + 15) / 16 * 16 + 4) * 4; }
// Sixteen rows of up to 2,544 columns fit the LDS of a compute unit; W's entries are counted in 32 bits.
constexpr bool spmm_gemm_fits(int n_rows, int K, int N) {
  return K >= 4 && spmm_gemm_lds(n_rows, K) <= kMaxLds && (long long)K * N <= UINT_MAX;
}

}  // namespace tf
