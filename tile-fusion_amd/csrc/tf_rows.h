// How the row kernels (tf_rows.hip) deal a row's columns to lanes and XCDs.  Host rules without a HIP header, so that a
// test can enumerate which lane stores which column.
#pragma once
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

// spmm_gemm_kernel: rows of A X a workgroup holds in LDS, and the LDS they take (K columns in steps of 16, four floats behind
// each row).
constexpr int spmm_gemm_rows(int n_rows) { return n_rows < 24000 ? 16 : 64; }
constexpr long long spmm_gemm_lds(int n_rows, int K) { return spmm_gemm_rows(n_rows) * (((long long)K + 15) / 16 * 16 + 4) * 4; }
// Sixteen rows of up to 2,544 columns fit the LDS of a compute unit; W's entries are counted in 32 bits.
constexpr bool spmm_gemm_fits(int n_rows, int K, int N) {
  return K >= 4 && spmm_gemm_lds(n_rows, K) <= kMaxLds && (long long)K * N <= UINT_MAX;
}

}  // namespace tf
