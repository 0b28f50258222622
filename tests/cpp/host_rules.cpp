// Rules of dispatch, checked on the host: which lane of which workgroup stores which column, what fits LDS.  Compiled with the host
// sources by tests/test_host_rules.py; each argument names a check; exits 0 when all of them hold.
#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <functional>
#include <vector>
#include "tf_internal.h"
#include "tf_rows.h"
namespace tf {
static char g_err[512];
tf_status fail(tf_status code, const char *fmt, ...) { va_list ap; va_start(ap, fmt); vsnprintf(g_err, sizeof g_err, fmt, ap); va_end(ap); return code; }
int default_compute_units() { return 256; }
void release_device_schedule(DeviceSchedule *) {}
}  // namespace tf

// Every column of a row is stored, and one that is added to is stored in one pass of one workgroup only: in a pass all lanes of a
// row load Y before one of them stores.  As in spmm_rows_kernel, over all widths and the strides and sizes that slices look at.
static int column_owners() {
  int bad = 0, sliced = 0;
  for (int accumulate = 0; accumulate < 2; ++accumulate)
    for (int N = 1; N <= 600; ++N)
      for (int pad = 0; pad < 2; ++pad)
        for (int compact = 0; compact < 2; ++compact)
          for (unsigned rows : {100u, 16000u, 30000u, 70000u, 131072u, 200000u}) {
            tf::RowsArgs a;
            a.X = reinterpret_cast<const float *>(1 << 20);
            a.ldx = pad ? (N + 31) / 32 * 32 : N;
            a.x_rows = rows;
            a.N = N;
            a.compact = compact;
            a.accumulate = accumulate;
            tf::RowShape s = tf::row_shape(N, accumulate);
            a.slices = s.V == 4 ? tf::slices_for(a) : 1;
            if (a.slices > 1) { s.LPR = tf::kSliceCols / 4; ++sliced; }
            std::vector<int> passes(N, 0), last(N, -1);
            int pass = 0;
            for (int slice = 0; slice < a.slices; ++slice) {
              const int c_begin = a.slices > 1 ? slice * s.LPR * s.V : 0;
              const int c_end = a.slices > 1 ? (N < c_begin + s.LPR * s.V ? N : c_begin + s.LPR * s.V) : N;
              for (int c0 = c_begin; c0 < c_end; c0 += s.LPR * s.V, ++pass)
                for (int lane = 0; lane < s.LPR; ++lane) {
                  const int col = c0 + lane * s.V;
                  if (col >= N) continue;
                  const int at = s.V == 1 ? tf::clamp_col<1>(col, N) : tf::clamp_col<4>(col, N);
                  for (int u = 0; u < s.V; ++u) {
                    if (at + u < 0 || at + u >= N) { printf("N %d: column %d stored\n", N, at + u); ++bad; continue; }
                    if (last[at + u] != pass) { last[at + u] = pass; ++passes[at + u]; }
                  }
                }
            }
            for (int c = 0; c < N; ++c)
              if (passes[c] < 1 || (accumulate && passes[c] > 1)) {
                printf("N %d rows %u slices %d accumulate %d: column %d in %d passes\n", N, rows, a.slices, accumulate, c, passes[c]);
                ++bad;
              }
          }
  if (!sliced) { printf("no slices anywhere\n"); ++bad; }
  return bad;
}

// The same for sweep_rows_kernel: a lane group takes a slice's columns in one go, X is within the 32 bits of its offsets, and the limit is behind it
// after the steps.
static int sweep_columns() {
  int bad = 0, shapes[3] = {};
  for (int N = 1; N <= 140; ++N)
    for (long long rows : {1000LL, 29000LL, 30000LL, 60000LL, 90000LL, 125000LL, 300000LL, 1000000LL, 17000000LL})
      for (int ldx : {N, (N + 31) / 32 * 32})
        for (int off : {0, 16})
          for (int accumulate : {0, 1})
            for (int mean : {5, 6, 40}) {
              tf::RowsArgs a;
              tf::RowsHow how;
              a.X = reinterpret_cast<const float *>((uintptr_t)4096 + off);
              a.ldx = ldx; a.N = N; a.n_rows = (int)rows; a.x_rows = (unsigned)rows; a.accumulate = accumulate;
              how.spread_entries = rows * mean;
              const tf::SweepShape s = tf::sweep_for(a, how);
              if (s.LPR == 0) continue;
              ++shapes[s.slices / 2];
              std::vector<int> owners(N, 0);
              for (int slice = 0; slice < s.slices; ++slice) {
                std::vector<char> mine(N, 0);
                for (int lane = 0; lane < s.LPR; ++lane) {
                  const int col = slice * s.LPR * 4 + lane * 4;
                  if (col >= N) continue;
                  for (int u = 0; u < 4; ++u) mine[tf::clamp_col<4>(col, N) + u] = 1;
                }
                for (int c = 0; c < N; ++c) owners[c] += mine[c];
              }
              bool ok = (s.LPR == 4 || s.LPR == 8 || s.LPR == 16 || s.LPR == 32) && s.LPR * 4 * s.slices >= N && 8 % s.slices == 0 && mean >= 6;
              for (int c = 0; c < N; ++c) ok = ok && owners[c] >= 1 && (!accumulate || owners[c] == 1);
              const unsigned long long bytes = (unsigned long long)rows * ldx * 4, step = bytes / s.steps + 1;
              ok = ok && bytes <= 0x80000000ull && s.steps >= mean && step * s.steps >= bytes && step * s.steps < 0xffffffffull;
              if (!ok) { printf("N %d ldx %d rows %lld accumulate %d: %d lanes, %d slices, %d steps\n", N, ldx, rows, accumulate, s.LPR, s.slices, s.steps); ++bad; }
            }
  for (int n : shapes) bad += n == 0;
  // 128 columns: four slices of the other kernel up to 20 MB of X
  for (long long rows : {30000LL, 39000LL, 39104LL, 46000LL})
    for (int mean : {6, 11, 17})
      if (tf::sweep_fits(rows, 128, rows, rows * mean) != (rows > 39062)) { printf("%lld rows of %d, N 128\n", rows, mean); ++bad; }
  return bad;
}

// Layers that run in one launch: the rows of A B that a workgroup holds fit its LDS, at every K; wider ones are inspected into something
// else and accepted all the same.
static int one_launch_fits() {
  int bad = 0, taken = 0, beyond = 0;
  for (int M : {1, 17, 500, 786, 4096, 9999, 23999, 24000, 30000}) {
    std::vector<int> p(M + 1), i;
    for (int r = 0; r < M; ++r) {
      for (int c = r > 0 ? r - 1 : 0; c <= r + 1 && c < M; ++c) i.push_back(c);
      p[r + 1] = (int)i.size();
    }
    for (int K : {4, 30, 64, 128, 250, 1000, 2543, 2544, 2545, 2560, 3000, 5000})
      for (int N : {2, 64, 128, 700, 1273, 2000, 2600}) {
        if ((long long)M * K > 4000000) continue;
        tf_inspect_opts o{};
        o.struct_size = sizeof(o);
        o.op = TF_OP_GEMM_SPMM;
        o.K = K;
        o.N = N;
        tf_schedule *s = nullptr;
        if (tf_inspect(M, M, p.data(), i.data(), &o, &s)) { printf("M %d K %d N %d: %s\n", M, K, N, tf::g_err); ++bad; continue; }
        if (tf_schedule_validate(s, M, M, p.data(), i.data())) { printf("M %d K %d N %d: %s\n", M, K, N, tf::g_err); ++bad; }
        const int lds = s->one_launch ? (s->two_passes->rem_rows.size() < 24000 ? 16 : 64) * ((K + 15) / 16 * 16 + 4) * 4 : 0;
        if (lds > 163840) { printf("M %d K %d N %d: one launch with %d bytes of LDS\n", M, K, N, lds); ++bad; }
        taken += s->one_launch;
        beyond += K > 2544 && K <= 2 * N && (long long)M * K <= 2000000;
        tf_schedule_free(s);
      }
  }
  if (!taken || !beyond) { printf("one launch %d times, %d sizes beyond it\n", taken, beyond); ++bad; }
  return bad;
}

// The row products of a schedule have room for partial sums of the width they run at, also on a band with hub rows, where the order of
// the products is chosen again.
static int partial_sums() {
  int bad = 0, again = 0;
  for (int M : {3000, 9000, 30000}) {
    std::vector<int> p(1, 0), i;
    for (int r = 0; r < M; ++r) {
      if (r % 1000 == 500) for (int c = r % 2; c < M; c += 2) i.push_back(c);
      else for (int c = r > 8 ? r - 8 : 0; c <= r + 8 && c < M; ++c) i.push_back(c);
      p.push_back((int)i.size());
    }
    for (int K : {8, 30, 32, 64, 100, 128})
      for (int N : {7, 32, 40, 64, 80, 96, 128, 140}) {
        tf_inspect_opts o{};
        o.struct_size = sizeof(o);
        o.op = TF_OP_GEMM_SPMM;
        o.K = K;
        o.N = N;
        tf_schedule *s = nullptr;
        if (tf_inspect(M, M, p.data(), i.data(), &o, &s)) { printf("M %d K %d N %d: %s\n", M, K, N, tf::g_err); ++bad; continue; }
        if (tf_schedule_validate(s, M, M, p.data(), i.data())) { printf("M %d K %d N %d: %s\n", M, K, N, tf::g_err); ++bad; }
        if (const tf_schedule *rows = s->two_passes) {
          const int width = s->spmm_first ? K : N;
          if (rows->opts.N < width) { printf("M %d K %d N %d: partial sums of %d columns for a product of %d\n", M, K, N, rows->opts.N, width); ++bad; }
          again += !s->spmm_first && K >= 4 && M < 10000 && N > K;
        }
        tf_schedule_free(s);
      }
  }
  if (!again) { printf("the order is never chosen again\n"); ++bad; }
  return bad;
}

// Hub rows that end the choice of one launch are seen before its lists are made; rows near the lengths where lists differ are not
// taken for them.  And columns out of range are refused by both inspectors, wherever in a row they stand.
static int hubs_and_columns() {
  int bad = 0;
  const int M = 6000;
  for (int longest : {31, 32, 33, 64, 65, 127, 128, 129, 1025})
    for (int K : {64, 30})
      for (int N : {64, 40, 20}) {
        std::vector<int> p(1, 0), i;
        for (int r = 0; r < M; ++r) {
          const int len = r == 3000 ? longest : 3;
          for (int k = 0; k < len; ++k) i.push_back((r + k * 3) % M);
          p.push_back((int)i.size());
        }
        tf_inspect_opts o{};
        o.struct_size = sizeof(o);
        o.op = TF_OP_GEMM_SPMM;
        o.K = K;
        o.N = N;
        tf_schedule *s = nullptr, *rows = nullptr;
        if (tf_inspect(M, M, p.data(), i.data(), &o, &s) || tf_inspect_spmm(M, M, p.data(), i.data(), K, 0, &rows)) { printf("%s\n", tf::g_err); return 1; }
        if (tf_schedule_validate(s, M, M, p.data(), i.data()) || tf_schedule_validate(rows, M, M, p.data(), i.data())) { printf("%s\n", tf::g_err); ++bad; }
        const bool cut = !rows->long_chunks.empty();
        if (cut != (longest > 32) || (s->one_launch && cut) || (!cut && !s->one_launch) || (cut && s->spmm_first != (3 * K <= 2 * N)) ||
            (s->two_passes && s->two_passes->opts.N < (s->spmm_first ? K : N))) {
          printf("longest %d K %d N %d: one launch %d, (A B) C %d\n", longest, K, N, s->one_launch, s->spmm_first);
          ++bad;
        }
        tf_schedule_free(s);
        tf_schedule_free(rows);
        for (int at : {0, 8999, 9000 + longest - 1, (int)i.size() - 1})
          for (int c : {-1, INT_MIN, M, INT_MAX}) {
            const int was = i[at];
            i[at] = c;
            if (tf_inspect(M, M, p.data(), i.data(), &o, &s) != TF_EINVAL || tf_inspect_spmm(M, M, p.data(), i.data(), N, 0, &rows) != TF_EINVAL) { printf("column %d accepted\n", c); ++bad; }
            i[at] = was;
          }
      }
  return bad;
}

// Streamed GeMM-SpMM runs: the last lane group's reads of a row's entries end inside the LDS that the kernel is launched with, and every
// quarter (half) of a group's slots is read by the lane of a quad that it is passed on from.
static int streamed_entries() {
  int bad = 0, streamed = 0;
  const int M = 30000;
  std::vector<int> p(M + 1), i;
  for (int r = 0; r < M; ++r) {
    for (int c = r > 2 ? r - 3 : 0; c <= r + 3 && c < M; ++c) i.push_back(c);
    p[r + 1] = (int)i.size();
  }
  for (int N : {32, 64, 96, 128})
    for (int K : {8, 64, 128, 136, 256})
      for (int budget : {65536, 102400, 163840}) {
        tf_inspect_opts o{};
        o.struct_size = sizeof(o);
        o.op = TF_OP_GEMM_SPMM;
        o.K = K;
        o.N = N;
        o.lds_budget_bytes = budget;
        tf_schedule *s = nullptr;
        if (tf_inspect(M, M, p.data(), i.data(), &o, &s)) { printf("%s\n", tf::g_err); return 1; }
        if (s->gemm_stream) {
          ++streamed;
          const int lanes = N <= 32 ? 8 : N <= 64 ? 16 : 32, consumers = K <= 128 ? 8 : 4;
          const long long scratch = tf::kStreamStageBytes + (long long)s->ring_rows * (N + 4) * 4;
          for (int g = 0; g < consumers * 64 / lanes; ++g)
            for (int l = 0; l < lanes; ++l) {
              const int q = tf::stream_quarter(l, lanes);
              for (int c = 0; c < lanes; c += 16) {
                const int slot = c + 4 * q + 3;  // of the group's
                if (slot >= lanes || scratch + 8LL * (g * lanes + slot + 1) > s->lds_bytes) {
                  printf("N %d K %d budget %d: lane %d of group %d reads slot %d, LDS ends at %d\n", N, K, budget, l, g, slot, s->lds_bytes);
                  ++bad;
                }
              }
              if (4 * (l & 3) < lanes && q != (l & 3)) { printf("lane %d of %d reads quarter %d\n", l, lanes, q); ++bad; }
            }
        }
        tf_schedule_free(s);
      }
  if (streamed < 20) { printf("%d streamed\n", streamed); ++bad; }
  return bad;
}

// Graphs whose reads are spread alike take the sweep, in one product as in two; one column that is read 255 times or more and they do not, whatever
// a byte makes of its count.  Nor do rows whose columns are in no order, or fall.
static int even_reads() {
  int bad = 0;
  const int M = 60000, mean = 11;
  for (int order = 0; order < 3; ++order)
    for (int often : {0, 254, 255, 256, 257, 300, 512, 767, 1024, 60000}) {
      std::vector<int> p(1, 0), i;
      unsigned long long at = 1;
      for (int r = 0; r < M; ++r) {
        for (int k = 0; k < mean; ++k) {
          at = at * 6364136223846793005ull + 1442695040888963407ull;
          i.push_back(1 + (int)((at >> 33) % (M - 1)));
        }
        if (r < often) i.push_back(0);
        if (order == 0) std::sort(i.begin() + p.back(), i.end());
        if (order == 1) std::sort(i.begin() + p.back(), i.end(), std::greater<int>());
        p.push_back((int)i.size());
      }
      const bool sweeps = often < 255 && order == 0;
      tf_inspect_opts o{};
      o.struct_size = sizeof(o);
      o.op = TF_OP_SPMM_SPMM;
      o.N = 64;
      tf_schedule *s = nullptr, *rows = nullptr;
      if (tf_inspect(M, M, p.data(), i.data(), &o, &s) || tf_inspect_spmm(M, M, p.data(), i.data(), 64, 0, &rows)) { printf("%s\n", tf::g_err); return 1; }
      if (!s->two_passes || s->two_passes->rem_sweep != sweeps || rows->rem_sweep != sweeps) { printf("order %d, a column read %d times\n", order, often); ++bad; }
      tf_schedule_free(s);
      tf_schedule_free(rows);
    }
  return bad;
}

// Far from the diagonal is not spread: rows that read where their neighbours in the order do, in blocks elsewhere, along another diagonal or in a part of their
// entries, have what a sweep would bring together.
static int rows_with_neighbours() {
  int bad = 0;
  const int M = 60000, mean = 11;
  unsigned long long at = 1;
  auto any = [&](int n) {
    at = at * 6364136223846793005ull + 1442695040888963407ull;
    return (int)((at >> 33) % n);
  };
  struct Kind { const char *name; int local, block, fields; bool sweep; };  // of 100 entries so many near the diagonal, blocks so large elsewhere, fields
  for (const Kind &kind : {Kind{"any", 0, M, 0, true}, Kind{"a quarter near", 25, M, 0, true}, Kind{"two thirds near", 67, M, 0, false}, Kind{"blocks of a sixth", 0, M / 6, 0, false},
                           Kind{"halves", 0, M / 2, 0, false}, Kind{"half near", 50, M, 0, true},
                           Kind{"blocks of 200", 0, 200, 0, false}, Kind{"two fields", 0, M, 2, false}, Kind{"three fields", 0, M, 3, false}}) {
    std::vector<int> p(1, 0), i;
    for (int r = 0; r < M; ++r) {
      const int base = (r / kind.block + M / kind.block / 2) % (M / kind.block) * kind.block;
      for (int k = 0; k < mean; ++k)
        i.push_back(kind.fields ? (r + M / kind.fields * (k % kind.fields) + k / kind.fields * 3) % M
                    : any(100) < kind.local ? std::min(M - 1, std::max(0, r + any(33) - 16)) : base + any(kind.block));
      std::sort(i.begin() + p.back(), i.end());
      p.push_back((int)i.size());
    }
    tf_schedule *rows = nullptr;
    if (tf_inspect_spmm(M, M, p.data(), i.data(), 64, 0, &rows)) { printf("%s\n", tf::g_err); return 1; }
    if (rows->rem_sweep != kind.sweep) { printf("%s\n", kind.name); ++bad; }
    tf_schedule_free(rows);
  }
  return bad;
}

int main(int argc, char **argv) {
  int bad = 0;
  for (int k = 1; k < argc; ++k) {
    const int b = !strcmp(argv[k], "column_owners") ? column_owners() : !strcmp(argv[k], "sweep_columns") ? sweep_columns() : !strcmp(argv[k], "one_launch_fits") ? one_launch_fits()
                  : !strcmp(argv[k], "partial_sums") ? partial_sums()
                  : !strcmp(argv[k], "hubs_and_columns") ? hubs_and_columns()
                  : !strcmp(argv[k], "streamed_entries") ? streamed_entries()
                  : !strcmp(argv[k], "even_reads") ? even_reads()
                  : !strcmp(argv[k], "rows_with_neighbours") ? rows_with_neighbours() : 1;
    printf("%s: bad %d\n", argv[k], b);
    bad += b;
  }
  return bad != 0;
}
