// Dense products beside the two executors: Y = X W for any K, N and either storage of W, and the gradient of a
// layer's weights, Y = G^T X, a product of small size summed over all rows.  Written for gfx950, fp32 MFMA.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <climits>

#include "tf_internal.h"
#include "tf_device.h"

namespace tf {

typedef float acc16 __attribute__((ext_vector_type(16)));

// ---------------------------------------------------------------------------------
// Y[q, :N] = X[rows[q], :K] * W, W stored K x N or (WT) N x K as torch stores a layer's weights, any K and N.
// A wavefront owns 16 rows and 16 CB columns of v_mfma_f32_16x16x4_f32; KW wavefronts of a workgroup share a row
// tile and take every KW-th step of 16 values of k each (their sums are added through LDS in a fixed order), so that
// a product of few rows still fills the device: 3,000 rows x 500 x 32 are 376 workgroups whose wavefronts have 8
// steps each, where one 32-row block per wavefront with all of K is 94 wavefronts of 250 MFMAs in a chain
// (13.2 us; 6.9 us here).  X and W come straight from global memory -- the wavefronts of a workgroup read the same W, which L1
// serves -- with k permuted inside a step the same way for both operands: lane (j, h) holds k = 16 s + 4 h + t for
// MFMA t, one 16-byte load of X, and of W when it is stored N x K.  Columns are dealt to lanes CB at a time
// (column CB j + cb to column block cb), so that a K x N stored W is loaded, and Y stored, CB floats per lane.
// ---------------------------------------------------------------------------------
template <int CB, int KW, bool WT>
__global__ __launch_bounds__(256) void gemm_direct_kernel(const float *__restrict__ X, int ldx, const float *__restrict__ W,
                                                          float *__restrict__ Y, int ldy, const int *__restrict__ rows,
                                                          int y_by_row, int n_rows, int K, int N,
                                                          const GemmOut out_how) {
  constexpr int RT = 4 / KW;  // row tiles per workgroup
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, j = lane % 16, h = lane / 16;
  const int kw = wave % KW, rt = wave / KW;
  const int row0 = (blockIdx.x * RT + rt) * 16, col0 = blockIdx.y * 16 * CB + CB * j;
  const int q = min(row0 + j, n_rows - 1);
  const float *xp = X + (size_t)(rows ? rows[q] : q) * ldx + 4 * h;
  const float *wp[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const int c = min(col0 + cb, N - 1);
    wp[cb] = WT ? W + (size_t)c * K + 4 * h : W + (size_t)(4 * h) * N + c;
  }
  const bool whole = col0 + CB <= N;  // this lane's CB columns exist
  acc4 acc[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) acc[cb] = 0.f;
  struct operands { f4v a, b[CB]; };
  auto load = [&](int s) __attribute__((always_inline)) {
    operands o;
    o.a = *reinterpret_cast<const f4u *>(xp + 16 * s);
    if constexpr (WT) {
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) o.b[cb] = *reinterpret_cast<const f4u *>(wp[cb] + 16 * s);
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const size_t at = (size_t)(16 * s + t) * N;
        if (whole) {
          const cvec<CB> w = *reinterpret_cast<const cvec<CB> *>(wp[0] + at);
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) o.b[cb][t] = w.v[cb];
        } else {
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) o.b[cb][t] = wp[cb][at];
        }
      }
    }
    return o;
  };
  auto multiply = [&](const operands &o) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) acc[cb] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.a[t], o.b[cb][t], acc[cb], 0, 0, 0);
  };
  const int full = K / 16;
  if (kw < full) {
    operands cur = load(kw);
    for (int s = kw; s < full; s += KW) {
      const operands nxt = load(min(s + KW, full - 1));
      multiply(cur);
      cur = nxt;
    }
  }
  if (K % 16 != 0 && full % KW == kw) {  // the last step: values of k past K are zeros in both operands
    operands o;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bool in = 16 * full + 4 * h + t < K;
      o.a[t] = in ? xp[16 * full + t] : 0.f;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) o.b[cb][t] = in ? (WT ? wp[cb][16 * full + t] : wp[cb][(size_t)(16 * full + t) * N]) : 0.f;
    }
    multiply(o);
  }
  if constexpr (KW > 1) {
    __shared__ acc4 part[RT][KW - 1][CB][64];
    if (kw > 0) {
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) part[rt][kw - 1][cb][lane] = acc[cb];
    }
    __syncthreads();
    if (kw > 0) return;
#pragma unroll
    for (int w = 0; w < KW - 1; ++w)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) acc[cb] += part[rt][w][cb][lane];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {  // register r of lane (j, h): row 4 h + r of the tile
    const int x = row0 + 4 * h + r;
    if (x >= n_rows) continue;
    const size_t at = (size_t)(rows && y_by_row ? rows[x] : x) * ldy + col0;
    cvec<CB> out;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) out.v[cb] = acc[cb][r];
    gemm_store<CB>(Y, at, out, N - col0, out_how);
  }
}

// ---------------------------------------------------------------------------------
// The same product for many rows: W (a panel of 16 V Q columns of it) in LDS, once per workgroup, row-major and padded with zeros
// to whole steps of k and whole panels, whichever way it is stored; every wavefront takes 16-row blocks
// with no barrier, its rows of X requested a group of A steps ahead (the first group before W is staged).
// Column block (v, q) of lane j is column 16 V q + V j + v: a lane reads V adjacent values of W per k and stores V adjacent columns of
// Y, sixteen lanes side by side.  Sixteen wavefronts per compute unit (up to 128 registers each), so that a SIMD has
// three others to feed its matrix core while one waits: 131,072 x 300 x 64 takes 54 us (139 us with
// every row tile reading W from L2; 33 us and 39 us for a padded copy of X in 32-row blocks).
// The wavefronts take blocks in turn, so that what is read and written is one stretch of memory; with K of 16 or less a group is the one step there is.
// (us, 262,144 rows, a kernel of 32-row MFMAs that took such rows before this one / a run of blocks for each wavefront / in turn / and one step:
// 8 x 32 12.7 / 13.7 / 13.0 / 11.9, 64 x 32 24.5 / 24.7 / 20.5, 8 x 64 17.7 / 20.2 / 19.0 / 18.0, 16 x 64 20.8 / 23.0 / 19.9 / 18.7, 8 x 128 29.5 / 35.8 / 33.4 / 30.2,
// 16 x 128 32.2 / 42.0 / 35.9 / 31.2, 128 x 32 40.5 / 40.7 / 34.2; 1,000,000 rows 16 x 128 124 / 140 / 140 / 118; 16,000 rows 128 x 128 12.0 / 11.9 / 11.4.)
// Bound: X and Y from HBM for up to 64 columns, fp32 MFMA beyond.
// ---------------------------------------------------------------------------------
constexpr int kGemmAhead = 4;  // A: steps of 16 values of k per group of operands

// Rows in order and values as they are; with zeros where the mask is zero or less; rows of a list, values as they are; all else.
enum { kPlain, kMasked, kListed, kAnyOut };

// The loop has no load or store under a condition, so that a wait for a group of operands leaves younger requests and the
// stores before them in flight: rows past the last one are the last one again and store its values once more, a lane whose
// V columns reach past the last one works on the last V, and the last step's values of k past K are cleared in registers.
// (Conditions around them, us: 262,144 x 64 x 64 37, 128 x 64 58, 64 x 128 61; without 29, 50, 55;
// 30,000 x 300 x 64 23.0, 100 x 83 15.8; without 18.3, 13.1.)
template <int V, int Q, bool WT, int OUT, int A>
__global__ __launch_bounds__(1024) void gemm_panel_kernel(const float *__restrict__ X, int ldx, const float *__restrict__ W,
                                                          float *__restrict__ Y, int ldy, const int *__restrict__ rows,
                                                          int y_by_row, int n_rows, int K, int N,
                                                          const GemmOut out_how) {
  extern __shared__ __align__(16) float wlds[];
  constexpr int P = 16 * V * Q;  // columns of the panel
  const int waves = blockDim.x / 64, wave = threadIdx.x / 64, lane = threadIdx.x % 64, j = lane % 16, h = lane / 16;
  const int panel0 = blockIdx.y * P, S = (K + 15) / 16, G = (S + A - 1) / A;
  const int n_blocks = (n_rows + 15) / 16, stride = gridDim.x * waves, b0 = wave * gridDim.x + blockIdx.x;
  auto column = [&](int n) { return OUT == kAnyOut ? min(panel0 + n, N - 1) : min(panel0 + n - n % V, N - V) + n % V; };  // of W
  struct operands { f4v a[A]; };
  auto row_index = [&](int b) __attribute__((always_inline)) {
    const int q = min(b * 16 + j, n_rows - 1);
    if constexpr (OUT == kPlain || OUT == kMasked) return q;
    else if constexpr (OUT == kListed) return rows[q];
    else return rows ? rows[q] : q;
  };
  auto load = [&](const float *xp, int g) __attribute__((always_inline)) {
    operands o;
#pragma unroll
    for (int u = 0; u < A; ++u) o.a[u] = *reinterpret_cast<const f4u *>(xp + min(16 * (g * A + u) + 4 * h, K - 4));
    return o;
  };
  const float *xp = X;
  operands cur;
  int next_row = 0;  // of this lane in the block after the next one to begin
  if (b0 < n_blocks) {
    xp = X + (size_t)row_index(b0) * ldx;
    next_row = row_index(b0 + stride);
    cur = load(xp, 0);
  }
  // W into LDS: a column's sixteen values of one step per thread and item, all requested before the first is stored
  for (int it = threadIdx.x; it < S * P; it += blockDim.x) {
    const int n = it % P, s = it / P, c = column(n);
    f4v v[4];
    if (16 * s + 16 <= K) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if constexpr (WT) v[u] = *reinterpret_cast<const f4u *>(W + (size_t)c * K + 16 * s + 4 * u);
        else {
#pragma unroll
          for (int t = 0; t < 4; ++t) v[u][t] = W[(size_t)(16 * s + 4 * u + t) * N + c];
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int k = 16 * s + 4 * u + t;
          v[u][t] = k < K ? (WT ? W[(size_t)c * K + k] : W[(size_t)k * N + c]) : 0.f;
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int t = 0; t < 4; ++t) wlds[(16 * s + 4 * u + t) * P + n] = v[u][t];
  }
  __syncthreads();
  acc4 acc[Q][V];
  const float *wl = wlds + 4 * h * P + V * j;
  auto step = [&](int s, const f4v &a) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float *w = wl + (16 * s + t) * P;
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        typedef float wv __attribute__((ext_vector_type(V)));
        wv b;
        if constexpr (V == 1) b[0] = w[16 * q]; else b = *reinterpret_cast<const wv *>(w + 16 * V * q);
#pragma unroll
        for (int v = 0; v < V; ++v) acc[q][v] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], b[v], acc[q][v], 0, 0, 0);
      }
    }
  };
  auto run = [&](int g, const operands &o) __attribute__((always_inline)) {
    if (16 * A * (g + 1) <= K) {
#pragma unroll
      for (int u = 0; u < A; ++u) step(g * A + u, o.a[u]);
      return;
    }
#pragma unroll
    for (int u = 0; u < A; ++u) {
      const int s = g * A + u, at = 16 * s + 4 * h, d = at - min(at, K - 4);
      if (s >= S) break;
      // the step's values are d places behind those that were loaded, zeros follow
      f4v v = o.a[u];
      v = d & 1 ? f4v{v[1], v[2], v[3], 0.f} : v;
      v = d & 2 ? f4v{v[2], v[3], 0.f, 0.f} : v;
      v = d >= 4 ? f4v{0.f, 0.f, 0.f, 0.f} : v;
      step(s, v);
    }
  };
  for (int b = b0; b < n_blocks; b += stride) {
    const float *xn = X + (size_t)next_row * ldx;
    next_row = row_index(b + 2 * stride);
    int y_row[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int x = min(b * 16 + 4 * h + r, n_rows - 1);
      if constexpr (OUT == kListed) y_row[r] = rows[x]; else y_row[r] = x;
      if (OUT == kListed && !y_by_row) y_row[r] = x;
    }
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int v = 0; v < V; ++v) acc[q][v] = 0.f;
    for (int g = 0; g < G; ++g) {
      operands nxt = load(g + 1 < G ? xp : xn, g + 1 < G ? g + 1 : 0);
      run(g, cur);
      cur = nxt;
    }
    xp = xn;
    if constexpr (OUT == kAnyOut) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int x = b * 16 + 4 * h + r;
        if (x >= n_rows) continue;
        const size_t row = (size_t)(rows && y_by_row ? rows[x] : x) * ldy;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          const int c = panel0 + 16 * V * q + V * j;
          cvec<V> out;
#pragma unroll
          for (int v = 0; v < V; ++v) out.v[v] = acc[q][v][r];
          gemm_store<V>(Y, row + c, out, N - c, out_how);
        }
      }
    } else {
      size_t at[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) at[r] = (size_t)y_row[r] * ldy;
      cvec<V> m[4][Q];
      if constexpr (OUT == kMasked) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int q = 0; q < Q; ++q) m[r][q] = *reinterpret_cast<const cvec<V> *>(out_how.mask + at[r] + min(panel0 + 16 * V * q + V * j, N - V));
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          cvec<V> out;
#pragma unroll
          for (int v = 0; v < V; ++v) out.v[v] = OUT == kMasked && m[r][q].v[v] <= 0.f ? 0.f : acc[q][v][r];
          *reinterpret_cast<cvec<V> *>(Y + at[r] + min(panel0 + 16 * V * q + V * j, N - V)) = out;
        }
    }
  }
}

// ---------------------------------------------------------------------------------
// The same on the bf16 matrix cores (split8 in tf_device.h), for W whose three bf16 parts fit LDS: a step is 32 values of k, W's parts lie
// in LDS as the matrix cores take them (a lane's eight values of a column in one 16-byte read), X's are made in registers on
// the way.  Bound: X and Y from HBM behind some 8 us until the first product (262,144 x 128 x 128 84 us in turn with other
// operands, gemm_panel_kernel 98, waiting for the fp32 cores; 63 and 81 with six products on a cooler board), and the board's power: the same on operands that are all the
// same number runs at 5.2 TB/s, and two tiles' products side by side change nothing.  Where W takes two panels the parts of X are made twice:
// 200,000 x 256 x 128 106 us, 60 at the rate of a copy.
// What is not finite: a row of X costs its block a second pass on the fp32 cores (100,000 x 128 x 128 39.4 -> 39.6 us, 131,072 x 300 x 64 51.8 -> 58.7; with
// one load at a time 36 -> 63 and 52 -> 91), a value in W one for every block: 79 and 125 us, 335 where W is N x K (176, 345, 415; a product on
// the fp32 cores alone 45 and 57).
// ---------------------------------------------------------------------------------
// Eight wavefronts per compute unit: more of them in flight read memory more slowly (100,000 x 300 x 64: 41.5 us, twelve 41.8, six 42.3).
constexpr int kSplitWaves = 8;
constexpr long long split_lds(int K, int columns) { return ((long long)K + 31) / 32 * columns * 192; }

template <int V, int Q, bool WT, int OUT, int A>
__global__ __launch_bounds__(64 * kSplitWaves) void gemm_split_kernel(const float *__restrict__ X, int ldx, const float *__restrict__ W,
                                                                   float *__restrict__ Y, int ldy, const int *__restrict__ rows,
                                                                   int y_by_row, int n_rows, int K, int N,
                                                                   const GemmOut out_how) {
  extern __shared__ __align__(16) bf8 wparts[];  // [step][tile][part][lane]
  constexpr int P = 16 * V * Q, T = V * Q;
  const int waves = blockDim.x / 64, wave = threadIdx.x / 64, lane = threadIdx.x % 64, j = lane % 16, h = lane / 16;
  const int panel0 = blockIdx.y * P, S = (K + 31) / 32, G = (S + A - 1) / A;
  // Blocks in turn over the workgroups, so that what is being read is one stretch of memory and not a place per wavefront (reads alone,
  // 131,072 rows of 1 KB that no cache holds: 34.5 against 38.9 us).
  const int n_blocks = (n_rows + 15) / 16, stride = gridDim.x * waves, b0 = wave * gridDim.x + blockIdx.x;
  auto column = [&](int n) { return OUT == kAnyOut ? min(panel0 + n, N - 1) : min(panel0 + n - n % V, N - V) + n % V; };  // of W
  f4v x[A][2];  // a lane's eight values of the next A steps
  auto row_index = [&](int b) __attribute__((always_inline)) {
    const int q = min(b * 16 + j, n_rows - 1);
    if constexpr (OUT == kPlain || OUT == kMasked) return q;
    else if constexpr (OUT == kListed) return rows[q];
    else return rows ? rows[q] : q;
  };
  auto load = [&](const float *xp, int s, f4v (&o)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int w = 0; w < 2; ++w) o[w] = *reinterpret_cast<const f4u *>(xp + min(32 * s + 8 * h + 4 * w, K - 4));
  };
  // W's parts into LDS: a column's eight values of k per item, U items' loads on their way at a time, the first of them in front of
  // the first rows of X (loads return in order, and all workgroups' first rows are a burst of 16 MB).
  constexpr int U = 8;
  const int items = S * T * 64;
  f4v v[U][2];
  auto load_items = [&](int it0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int it = it0 + u * (int)blockDim.x;
      if (it >= items) break;  // (whole wavefronts: the items are a multiple of 64)
      const int jj = it % 16, hh = it / 16 % 4, t = it / 64 % T, s = it / (64 * T), k0 = 32 * s + 8 * hh;
      const int c = column(16 * V * (t / V) + V * jj + t % V);
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const int kk = k0 + 4 * w;
        if (kk + 4 <= K) {
          if constexpr (WT) v[u][w] = *reinterpret_cast<const f4u *>(W + (size_t)c * K + kk);
          else {
#pragma unroll
            for (int i = 0; i < 4; ++i) v[u][w][i] = W[(size_t)(kk + i) * N + c];
          }
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) v[u][w][i] = kk + i < K ? W[WT ? (size_t)c * K + kk + i : (size_t)(kk + i) * N + c] : 0.f;
        }
      }
    }
  };
  auto put_items = [&](int it0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int it = it0 + u * (int)blockDim.x;
      if (it >= items) break;
      const split3<bf8> p = split8(v[u][0], v[u][1]);
      bf8 *at = wparts + (size_t)(it / 64) * 192 + it % 64;
      at[0] = p.h;
      at[64] = p.m;
      at[128] = p.l;
    }
  };
  load_items(threadIdx.x);
  const float *xp = X;
  int row = 0, next_row = 0;  // of this lane in the block to begin next and in the one behind it
  if (b0 < n_blocks) {
    row = row_index(b0);
    xp = X + (size_t)row * ldx;
    next_row = row_index(b0 + stride);
#pragma unroll
    for (int u = 0; u < A; ++u) load(xp, u, x[u]);
  }
  put_items(threadIdx.x);
  for (int it0 = threadIdx.x + U * blockDim.x; it0 < items; it0 += U * blockDim.x) {
    load_items(it0);
    put_items(it0);
  }
  __syncthreads();
  acc4 big[T], small[T];
  const bf8 *wl = wparts + lane;
  auto multiply = [&](int s, const split3<bf8> &a) __attribute__((always_inline)) {
    const bf8 *w = wl + (size_t)s * (T * 192);
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const bf8 wh = w[t * 192], wm = w[t * 192 + 64], wlo = w[t * 192 + 128];
      small[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.l, wm, small[t], 0, 0, 0);
      small[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.m, wlo, small[t], 0, 0, 0);
      small[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.l, wh, small[t], 0, 0, 0);
      small[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, wlo, small[t], 0, 0, 0);
      small[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.m, wm, small[t], 0, 0, 0);
      small[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.m, wh, small[t], 0, 0, 0);
      small[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, wm, small[t], 0, 0, 0);
      big[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, wh, big[t], 0, 0, 0);
    }
  };
  // Where K is no multiple of four, one lane group's last values lie d places behind those that were loaded.  (W's parts are zero where k
  // is past K.)
  int d[2];
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    const int at = 32 * (S - 1) + 8 * h + 4 * w;
    d[w] = at < K ? at - min(at, K - 4) : 0;
  }
  // A step: its values become parts, whereupon their registers take the values A steps on, of this block or the next.
  auto step = [&](int s, f4v (&o)[2], const float *from, int ahead, float in_scale) __attribute__((always_inline)) {
    if (s == S - 1 && K % 4 != 0) {
      asm volatile("");  // (a branch: as selects these were 24 of a step's 138 vector instructions, 84 with split8's pairs)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        o[w] = d[w] & 1 ? f4v{o[w][1], o[w][2], o[w][3], 0.f} : o[w];
        o[w] = d[w] & 2 ? f4v{o[w][2], o[w][3], 0.f, 0.f} : o[w];
      }
    }
    const split3<bf8> a = split8(o[0], o[1], in_scale);
    load(from, ahead, o);
    __builtin_amdgcn_sched_barrier(0);  // (the requests stay in front of the products)
    if (s < S) multiply(s, a);
  };
  for (int b = b0; b < n_blocks; b += stride) {
    const float *xn = X + (size_t)next_row * ldx;
    const float in_scale = row & 1 ? -kSplitIn : kSplitIn;
    row = next_row;
    next_row = row_index(b + 2 * stride);
    int y_row[4];
    float out_scale[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int x = min(b * 16 + 4 * h + r, n_rows - 1);
      const int of = OUT == kPlain || OUT == kMasked ? x : OUT == kListed || rows ? rows[x] : x;
      y_row[r] = OUT == kListed && y_by_row ? of : x;
      out_scale[r] = of & 1 ? -kSplitOut : kSplitOut;
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
      big[t] = 0.f;
      small[t] = 0.f;
    }
    for (int g = 0; g < G; ++g) {
      const bool more = g + 1 < G;
#pragma unroll
      for (int u = 0; u < A; ++u) step(g * A + u, x[u], more ? xp : xn, more ? (g + 1) * A + u : u, in_scale);
    }
    float finite = 0.f;
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        big[t][r] = (big[t][r] + small[t][r]) * out_scale[r];
        finite = __builtin_fmaf(big[t][r], 0.f, finite);
      }
    if (__ballot(finite != 0.f)) {  // (NaN) infinities or NaN in the operands, or too large for bf16
#pragma unroll
      for (int t = 0; t < T; ++t) big[t] = 0.f;
#pragma unroll 1
      for (int k0 = 0; k0 < K; k0 += 16) {  // lane (j, h): values 4 h + u of sixteen in product u, all on their way at once
        float xv[4], wv[4][T];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int k = min(k0 + 4 * h + u, K - 1);
          xv[u] = xp[k];
#pragma unroll
          for (int t = 0; t < T; ++t) {
            const int c = column(16 * V * (t / V) + V * j + t % V);
            wv[u][t] = W[WT ? (size_t)c * K + k : (size_t)k * N + c];
          }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const bool in = k0 + 4 * h + u < K;
#pragma unroll
          for (int t = 0; t < T; ++t) big[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? xv[u] : 0.f, in ? wv[u][t] : 0.f, big[t], 0, 0, 0);
        }
      }
    }
    xp = xn;
    if constexpr (OUT == kAnyOut) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int x = b * 16 + 4 * h + r;
        if (x >= n_rows) continue;
        const size_t y = (size_t)(rows && y_by_row ? rows[x] : x) * ldy;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          const int c = panel0 + 16 * V * q + V * j;
          cvec<V> out;
#pragma unroll
          for (int v = 0; v < V; ++v) out.v[v] = big[q * V + v][r];
          gemm_store<V>(Y, y + c, out, N - c, out_how);
        }
      }
    } else {
      size_t at[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) at[r] = (size_t)y_row[r] * ldy;
      cvec<V> m[4][Q];
      if constexpr (OUT == kMasked) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int q = 0; q < Q; ++q) m[r][q] = *reinterpret_cast<const cvec<V> *>(out_how.mask + at[r] + min(panel0 + 16 * V * q + V * j, N - V));
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          cvec<V> out;
#pragma unroll
          for (int v = 0; v < V; ++v) out.v[v] = OUT == kMasked && m[r][q].v[v] <= 0.f ? 0.f : big[q * V + v][r];
          *reinterpret_cast<cvec<V> *>(Y + at[r] + min(panel0 + 16 * V * q + V * j, N - V)) = out;
        }
    }
  }
}

// X: n_rows x K, row stride ldx (or the rows of X that `rows` lists); Y: row q of it at q * ldy, or at rows[q] * ldy when
// y_by_row is set.  wt: W is N x K.
hipError_t launch_gemm_any(const float *X, int ldx, const float *W, int wt, float *Y, int ldy, const int *rows, int y_by_row,
                           int n_rows, int K, int N, const GemmOut &how, int compute_units, hipStream_t st) {
  if (n_rows <= 0) return hipSuccess;
  // Which kernel.  Copying W to LDS takes some 4 us before the first product; gemm_direct_kernel reads it from L2 for every row tile, by
  // single values where W is K x N (us, gemm_panel_kernel / gemm_direct_kernel, at 8,000 / 16,000 / 30,000 rows: 128 x 128 9.3 / 8.1 (K x N: 9.3 / 11.6),
  // 11.0 / 13.8, 16.8 / 23; 64 x 64 5.0 / 4.6 (5.0 / 5.7), 5.0 / 6.0, 6.7 / 9.0; 500 x 32, 30,000 rows 17.6 / 20.8; 40 x 7 6.7 / 4.2).
  // The bf16 cores pay where the fp32 ones are what a product waits for and panels of 64 columns fit LDS (up to 416 values of k): beyond 64 columns from 72
  // rows per compute unit on, where splitting W no longer counts (40 beyond 213 values of k, where a row block is a long chain of fp32
  // products), for 33 to 64 columns from 150 on where K is beyond 48 (us, gemm_panel_kernel / gemm_split_kernel, W as it is stored in turn: 10,240 rows
  // 192 x 128 13.8 / 16.8, 213 x 128 16.3 / 14.2, 14,000 rows 200 x 128 16.3 / 14.7, 213 x 96 14.4 / 15.3, 300 x 128 20.8 / 18.5; 18,432 rows 20 x 128 7.9 / 8.6, 32 x 128 8.1 / 7.4, 64 x 128 11.0 / 9.0, 128 x 128 16.2 / 14.9;
  // 20,000 rows 200 x 128 24.4 / 17.8; 30,000 rows 128 x 128 17.3 / 16.7; 60,000 rows 24 x 96 10.9 / 10.3, 128 x 128 26.6 / 23.9; 180,000 rows 24 x 128
  // 28.2 / 26.5; 38,400 rows 64 x 64 9.1 / 9.1, 128 x 64 12.9 / 13.5, 300 x 64 23.6 / 23.4; 40,000 rows 60 x 64 9.9 / 8.8; 60,000 rows 64 x 64 11.0 / 10.6;
  // 100,000 rows 49 x 64 15.3 / 15.1, 128 x 64 23.7 / 21.4, 300 x 64 47.7 / 40.5; 131,072 rows 60 x 40 18.4 / 15.5; 262,144 rows 64 x 64 28.1 / 27.0, 128 x 40
  // 45.0 / 39.4; five panels, 60,000 rows 300 x 300 169 / 93.  Panels of 32, where X is split for each: 40,000 rows 500 x 64 34.5 / 36.0, 100,000 rows
  // 73 / 77, 262,144 rows 165 / 181, 100,000 rows 832 x 48 108 / 122, 150,000 rows 512 x 128 173 / 194).
  // Widths are cut into equal panels that fit LDS; X is read once per panel, by compute units of the same XCD at about the same time.
  const int all_rows = std::max(n_rows, how.of_rows);
  bool on_bf16 = (N > 64 ? K > 16 && all_rows >= (K > 213 ? 40LL : 72LL) * compute_units : N > 32 && K > 48 && all_rows >= 150LL * compute_units) && split_lds(K, 64) <= kMaxLds;
  auto lds_of = [&](int columns) { return on_bf16 ? split_lds(K, columns) : ((long long)K + 15) / 16 * 16 * 4 * columns; };
  auto panel_width = [&]() {
    const int most = on_bf16 ? 128 : N <= 16 ? 16 : N <= 32 ? 32 : 128;
    const int panels0 = (N + most - 1) / most, w0 = (N + panels0 - 1) / panels0;
    int w = w0 <= 16 ? 16 : w0 <= 32 ? 32 : w0 <= 64 ? 64 : w0 <= 96 ? 96 : 128;
    while (w > (on_bf16 ? 64 : 16) && lds_of(w) > kMaxLds) w = w == 96 ? 64 : w / 2;
    return w;
  };
  int unit = panel_width();
  // (65 to 67 columns, of 257 values of k and more, are one panel of 96 on the fp32 cores, 60,000 rows 300 x 65 45 us, and one of 64 and the rest on the others, 51)
  if (on_bf16 && N > unit && N - unit < 4) {
    on_bf16 = false;
    unit = panel_width();
  }
  const long long from = N <= 16 ? LLONG_MAX : N <= 32 ? 80LL * compute_units : (wt ? 48LL : 24LL) * compute_units;
  if (all_rows >= from && lds_of(unit) <= kMaxLds && K >= 4) {
    const int panels = (N + unit - 1) / unit, lds = (int)lds_of(unit), n_blocks = (n_rows + 15) / 16;
    // workgroups per panel: a multiple of 8, so that a row block's panels are on one XCD
    const int across = on_bf16 ? std::max(8, compute_units / panels / 8 * 8) : compute_units / std::min(panels, 2);
    int waves = n_blocks >= 16 * compute_units ? 16 : n_blocks >= 8 * compute_units ? 8 : 4;
    // steps of k in flight: two, where three or five do not leave less of a rest of K's (us with two / three / four / five: 60,000 x 128 x 64 14.3 /
    // 15.9 / 15.9 / 16.0, 131,072 x 64 x 64 16.2 / 17.2 / 19.0 / 20.4, 300 x 64 48.5 / 51 / 50.5 / 48.6, 262,144 x 128 x 128 69.6 / 74.5 / 72 / 72.6, 30,000 x 300 x 128
    // 26.9 / 28.1 / 28.6 / 28.2; three steps of K, 100,000 x 96 x 128 29.2 / 27.7 / 28.8 / 29.4; five, 100,000 x 160 x 64 26.6 / 25.8 / 29.5 / 24.8)
    int ahead = 2;
    if (on_bf16) {
      waves = std::max(4, std::min(kSplitWaves, (n_blocks + across - 1) / across));
      const int steps = (K + 31) / 32;
      for (int n : {3, 5})
        if ((steps + n - 1) / n * n < (steps + ahead - 1) / ahead * ahead) ahead = n;
    }
    const dim3 grid(std::max(1, std::min(across, (n_blocks + waves - 1) / waves)), panels);
    hipError_t err = hipSuccess;
    // (a last panel of less than a lane's columns must not store the one before it: the two may differ in their last bits, where one of them went
    // over to the fp32 cores)
    const int lane_columns = unit == 16 ? 1 : unit % 64 ? 2 : 4;
    const bool narrow_last = on_bf16 && panels > 1 && N - (panels - 1) * unit < lane_columns;
    const int out = how.accumulate || how.relu || N < 4 || narrow_last || (rows && how.mask) ? kAnyOut : rows ? kListed : how.mask ? kMasked : kPlain;
#define CALLP4(...)                                                                                                            \
  do {                                                                                                                         \
    if (lds > 65536)                                                                                                           \
      err = hipFuncSetAttribute(reinterpret_cast<const void *>(__VA_ARGS__), hipFuncAttributeMaxDynamicSharedMemorySize, lds);  \
    if (err == hipSuccess)                                                                                                     \
      hipLaunchKernelGGL((__VA_ARGS__), grid, dim3(64 * waves), lds, st, X, ldx, W, Y, ldy, rows, y_by_row, n_rows, K, N, how); \
  } while (0)
#define CALLP3(V_, Q_, WT_, OUT_)                                                                                              \
  do {                                                                                                                         \
    if (!on_bf16 && K <= 16) { CALLP4(gemm_panel_kernel<V_, Q_, WT_, OUT_, 1>); }                                              \
    else if (!on_bf16) { CALLP4(gemm_panel_kernel<V_, Q_, WT_, OUT_, kGemmAhead>); }                                           \
    else if constexpr (V_ * Q_ >= 4) {                                                                                         \
      if (ahead == 5) { CALLP4(gemm_split_kernel<V_, Q_, WT_, OUT_, 5>); }                                                \
      else if (ahead == 3) { CALLP4(gemm_split_kernel<V_, Q_, WT_, OUT_, 3>); }                                                \
      else { CALLP4(gemm_split_kernel<V_, Q_, WT_, OUT_, 2>); }                                                                \
    }                                                                                                                          \
  } while (0)
#define CALLP2(V_, Q_, WT_)                                                                                                    \
  do { if (out == kPlain) { CALLP3(V_, Q_, WT_, kPlain); } else if (out == kMasked) { CALLP3(V_, Q_, WT_, kMasked); } else if (out == kListed) { CALLP3(V_, Q_, WT_, kListed); } else { CALLP3(V_, Q_, WT_, kAnyOut); } } while (0)
#define CALLP(V_, Q_) do { if (wt) { CALLP2(V_, Q_, true); } else { CALLP2(V_, Q_, false); } } while (0)
    switch (unit) {
      case 16: CALLP(1, 1); break;
      case 32: CALLP(2, 1); break;
      case 64: CALLP(4, 1); break;
      case 96: CALLP(2, 3); break;
      default: CALLP(4, 2); break;
    }
#undef CALLP
#undef CALLP2
#undef CALLP3
#undef CALLP4
    return err != hipSuccess ? err : hipGetLastError();
  }
  // Column blocks per wavefront: as many as the width has (up to four: X is then read once per 64 columns), fewer
  // where that leaves compute units without a workgroup.  Wavefronts per row tile: one when the row tiles fill the
  // device eight wavefronts deep, else the steps of k are shared out.
  const long long rt = (n_rows + 15) / 16;
  int cb = N > 32 ? 4 : N > 16 ? 2 : 1;
  while (cb > 1 && rt * ((N + 16 * cb - 1) / (16 * cb)) < compute_units) cb /= 2;
  const long long tiles = rt * ((N + 16 * cb - 1) / (16 * cb));
  const int kw = tiles >= 8LL * compute_units || K <= 32 ? 1 : tiles >= 4LL * compute_units || K <= 64 ? 2 : 4;
  const dim3 grid((unsigned)((rt + 4 / kw - 1) / (4 / kw)), (unsigned)((N + 16 * cb - 1) / (16 * cb)));
#define CALL3(CB_, KW_, WT_) \
  hipLaunchKernelGGL((gemm_direct_kernel<CB_, KW_, WT_>), grid, dim3(256), 0, st, X, ldx, W, Y, ldy, rows, y_by_row, n_rows, K, N, how)
#define CALL2(CB_, KW_) do { if (wt) { CALL3(CB_, KW_, true); } else { CALL3(CB_, KW_, false); } } while (0)
#define CALL(CB_) do { if (kw == 1) { CALL2(CB_, 1); } else if (kw == 2) { CALL2(CB_, 2); } else { CALL2(CB_, 4); } } while (0)
  if (cb == 4) CALL(4); else if (cb == 2) CALL(2); else CALL(1);
#undef CALL
#undef CALL2
#undef CALL3
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// Y[n, k] = sum over m < M of G[m, n] * X[m, k]: the gradient of a layer's weights, on the bf16 matrix cores (split8 in tf_device.h).  A
// wavefront holds a 16 NB x 16 KB tile of Y and takes 32 rows of both operands at a time, in whole lines: lane (j, h) loads the columns
// NB j .. of G and KB j .. of X in the rows 8 h .. 8 h + 7, which are what its part of a 16 x 16 x 32 product wants of each of
// the NB (KB) column blocks.  The next rows are requested as soon as these have become parts.  The wavefronts of a launch take blocks of
// rows in turn; a workgroup's four or eight are added through LDS, and weight_grad_reduce_kernel adds the workgroups' tiles -- all in a fixed order.
// A lane whose columns would reach past the last one works on the last NB (KB) instead: some values of Y are computed twice.
// Bound: the rows of X and G from HBM, 16 KB a wavefront in flight, behind some 10 us for two launches and the sums at the end (us, operands in no
// cache, both launches, fp32 cores on 64 x 160 tiles / this: 14,000 rows 32 x 69 18.0 / 10.3, 35,000 rows 64 x 128 25.7 / 22.8, 100,000 rows 64 x 128 36.3 / 32.0,
// 20 x 100 25.9 / 24.1, 131,072 rows 64 x 300 75 / 66, 40 x 64 28.1 / 26.0, 262,144 rows 128 x 128 105 / 94; relative error against 64 bits at 100,000 rows
// 1.8e-7 / 1.0e-7).
// ---------------------------------------------------------------------------------
constexpr int kWgRows = 32;       // rows of a block
constexpr int kWgFewRows = 4096;  // up to here in one launch, weight_grad_few_kernel

template <int NB, int KB, int WAVES>
__device__ __forceinline__ void weight_grad_tile(const WeightGradTask &t, int group, int chunk, acc4 (*red)[64]) {
  constexpr int T = NB * KB;
  const float *__restrict__ G = t.G, *__restrict__ X = t.X;
  const int N = t.N, K = t.K, M = t.M;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, j = lane % 16, h = lane / 16;
  const int nc = chunk / t.k_chunks, kc = chunk % t.k_chunks;
  const float *gp = G + min(nc * 16 * NB + NB * j, N - NB);
  const float *xp = X + min(kc * 16 * KB + KB * j, K - KB);
  const int n_blocks = (M + kWgRows - 1) / kWgRows, stride = WAVES * t.groups, b0 = WAVES * group + wave;
  acc4 acc[NB][KB];
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int b = 0; b < KB; ++b) acc[a][b] = 0.f;
  cvec<NB> g[8];
  cvec<KB> x[8];
  auto load_g = [&](int b) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) g[i] = *reinterpret_cast<const cvec<NB> *>(gp + (size_t)min(kWgRows * b + 8 * h + i, M - 1) * N);
  };
  auto load_x = [&](int b) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = *reinterpret_cast<const cvec<KB> *>(xp + (size_t)min(kWgRows * b + 8 * h + i, M - 1) * K);
  };
  if (b0 < n_blocks) {
    load_g(b0);
    load_x(b0);
  }
  for (int b = b0; b < n_blocks; b += stride) {
    if (kWgRows * (b + 1) > M) {  // rows past the last one are zeros in both operands
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (kWgRows * b + 8 * h + i >= M) {
#pragma unroll
          for (int a = 0; a < NB; ++a) g[i].v[a] = 0.f;
#pragma unroll
          for (int c = 0; c < KB; ++c) x[i].v[c] = 0.f;
        }
    }
    const float sign = b & 1 ? -1.f : 1.f;
    split3<bf8> gs[NB], xs[KB];
#pragma unroll
    for (int a = 0; a < NB; ++a) gs[a] = split8(f4v{g[0].v[a], g[1].v[a], g[2].v[a], g[3].v[a]}, f4v{g[4].v[a], g[5].v[a], g[6].v[a], g[7].v[a]}, sign * kSplitIn);
    load_g(b + stride);
#pragma unroll
    for (int c = 0; c < KB; ++c) xs[c] = split8(f4v{x[0].v[c], x[1].v[c], x[2].v[c], x[3].v[c]}, f4v{x[4].v[c], x[5].v[c], x[6].v[c], x[7].v[c]});
    load_x(b + stride);
    __builtin_amdgcn_sched_barrier(0);  // (the requests stay in front of the products)
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
      for (int c = 0; c < KB; ++c) {
        // The block's own sums, the large terms by themselves: h h of a few rows is exact, and what is left is rounded to nearest here, once per 32 rows.
        acc4 small = 0.f;
        small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gs[a].l, xs[c].m, small, 0, 0, 0);
        small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gs[a].m, xs[c].l, small, 0, 0, 0);
        small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gs[a].l, xs[c].h, small, 0, 0, 0);
        small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gs[a].h, xs[c].l, small, 0, 0, 0);
        small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gs[a].m, xs[c].m, small, 0, 0, 0);
        small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gs[a].m, xs[c].h, small, 0, 0, 0);
        small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gs[a].h, xs[c].m, small, 0, 0, 0);
        const acc4 big = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gs[a].h, xs[c].h, acc4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[a][c][r] = __builtin_fmaf(sign, big[r] + small[r], acc[a][c][r]);
      }
  }
  float finite = 0.f;
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int c = 0; c < KB; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        acc[a][c][r] *= kSplitOut;
        finite = __builtin_fmaf(acc[a][c][r], 0.f, finite);
      }
  if (__ballot(finite != 0.f)) {  // (NaN) infinities or NaN in the operands, or too large for the parts: on the fp32 cores
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
      for (int c = 0; c < KB; ++c) acc[a][c] = 0.f;
#pragma unroll 1
    for (int b = b0; b < n_blocks; b += stride)
#pragma unroll 1
      for (int m0 = kWgRows * b; m0 < min(kWgRows * (b + 1), M); m0 += 4) {
        const size_t m = min(m0 + h, M - 1);
        const float in = m0 + h < M ? 1.f : 0.f;
        cvec<NB> gv = *reinterpret_cast<const cvec<NB> *>(gp + m * N);
        cvec<KB> xv = *reinterpret_cast<const cvec<KB> *>(xp + m * K);
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
          for (int c = 0; c < KB; ++c)
            acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(in != 0.f ? gv.v[a] : 0.f, in != 0.f ? xv.v[c] : 0.f, acc[a][c], 0, 0, 0);
      }
  }
#pragma unroll
  for (int half = WAVES / 2; half >= 1; half /= 2) {
    if (wave >= half && wave < 2 * half) {
#pragma unroll
      for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int c = 0; c < KB; ++c) red[(wave - half) * T + a * KB + c][lane] = acc[a][c];
    }
    __syncthreads();
    if (wave < half) {
#pragma unroll
      for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int c = 0; c < KB; ++c) acc[a][c] += red[wave * T + a * KB + c][lane];
    }
    __syncthreads();
  }
  if (wave == 0) {  // partial[group][chunk][tile][register][lane]
    float *out = t.partial + ((size_t)group * (t.n_chunks * t.k_chunks) + chunk) * (T * 256) + lane;
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
      for (int c = 0; c < KB; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) out[((a * KB + c) * 4 + r) * 64] = acc[a][c][r];
  }
}

// Two gradients a launch: the workgroups from first_blocks on work on the second, whose rows come in while the first one's sums are added up.  (A
// training step of two layers on 13,800 nodes, 69 -> 32 -> 6: 17.7 us in four launches, 11.4 in two.)
template <int WAVES>
__global__ __launch_bounds__(64 * WAVES, 2) void weight_grad_kernel(const WeightGradTask first, const WeightGradTask second, int first_blocks) {
  __shared__ acc4 red[WAVES / 2 * 16][64];
  const bool other = (int)blockIdx.x >= first_blocks;
  const WeightGradTask &t = other ? second : first;
  const int at = other ? blockIdx.x - first_blocks : blockIdx.x, group = at % t.groups, chunk = at / t.groups;
#define TILE(NB_, KB_) case NB_ * 8 + KB_: weight_grad_tile<NB_, KB_, WAVES>(t, group, chunk, red); break
  switch (t.nb * 8 + t.kb) {
    TILE(1, 1); TILE(1, 2); TILE(1, 3); TILE(1, 4); TILE(2, 1); TILE(2, 2); TILE(2, 3); TILE(2, 4);
    TILE(3, 1); TILE(3, 2); TILE(3, 3); TILE(3, 4); TILE(4, 1); TILE(4, 2); TILE(4, 3); TILE(4, 4);
  }
#undef TILE
}

// Adds the groups' tiles: one workgroup per register of a tile, the groups dealt to its four wavefronts, eight loads of each in flight (four: 10 us
// for 256 groups of 64 x 128).
__global__ __launch_bounds__(256) void weight_grad_reduce_kernel(const WeightGradTask first, const WeightGradTask second, int first_blocks) {
  const bool other = (int)blockIdx.x >= first_blocks;
  const WeightGradTask &t = other ? second : first;
  const int at = other ? blockIdx.x - first_blocks : blockIdx.x, NB = t.nb, KB = t.kb, N = t.N, K = t.K, groups = t.groups, k_chunks = t.k_chunks;
  const int chunks = t.n_chunks * k_chunks;
  __shared__ float red[3][64];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, j = lane % 16, h = lane / 16;
  const int T = NB * KB, chunk = at / (4 * T), reg = at % (4 * T);
  const float *p = t.partial + (size_t)chunk * (T * 256) + reg * 64 + lane;
  const size_t stride = (size_t)chunks * (T * 256);
  float s = 0.f;
  for (int g = wave; g < groups; g += 32) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = p[(size_t)min(g + 4 * u, groups - 1) * stride];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = g + 4 * u < groups ? v[u] : 0.f;
    s += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
  }
  if (wave > 0) red[wave - 1][lane] = s;
  __syncthreads();
  if (wave > 0) return;
  s += red[0][lane];
  s += red[1][lane];
  s += red[2][lane];
  const int r = reg % 4, kb = (reg / 4) % KB, nb = reg / 4 / KB;
  const int i = 4 * h + r;  // row of the 16 x 16 block that register r of lane (j, h) holds
  const int n0 = chunk / k_chunks * 16 * NB, k0 = chunk % k_chunks * 16 * KB;
  const int n = min(n0 + NB * i, N - NB) + nb, k = min(k0 + KB * j, K - KB) + kb;
  // (what lies in front of the chunk is stored by the one it belongs to: the two may differ in their last bits, where one of them went over to the fp32 cores)
  if (n >= n0 && k >= k0) t.Y[(size_t)n * K + k] = s;
}

// The same for few rows in one launch: a workgroup of sixteen wavefronts per 16 x 16 tile of Y (v_mfma_f32_16x16x4_f32, so that
// there are tiles enough) and no partial sums in memory.  What counts is the chain of loads: a wavefront keeps sixteen steps of four
// rows in flight, eight being multiplied and the next eight on their way.  This / weight_grad_kernel and its sums, us: 16 x 40, 1,000 rows 5.8 / 7.4,
// 64 x 100, 2,000 rows 8.7 / 10.1, 7 x 32, 3,000 rows 8.0 / 7.0, 32 x 500, 3,000 rows 12.2 / 9.1, 32 x 100, 4,096 rows 14.3 / 7.9 -- and a launch and a
// workspace less for the host, which is what a small model waits for: 4,096 nodes, layer 100 -> 32 forward and backward 74 us (two launches 80), 512 -> 128 73
// (76), two layers 100 -> 32 -> 7 90 (94), 500 -> 64 -> 40 87 (93).
__global__ __launch_bounds__(1024, 4) void weight_grad_few_kernel(const WeightGradTask first, const WeightGradTask second, int first_blocks) {
  constexpr int W = 16, U = 8;
  __shared__ float red[W][4][64];
  const bool other = (int)blockIdx.x >= first_blocks;
  const WeightGradTask &t = other ? second : first;
  const float *__restrict__ G = t.G, *__restrict__ X = t.X;
  const int at = other ? blockIdx.x - first_blocks : blockIdx.x, N = t.N, K = t.K, M = t.M;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, j = lane % 16, h = lane / 16;
  const int n0 = at / t.k_chunks * 16, k0 = at % t.k_chunks * 16;
  // rows past the last one lie past the end of both buffers: their loads return zeros
  const __amdgpu_buffer_rsrc_t gr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(G), 0, M * N * 4, 0x00020000),
                               xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(X), 0, M * K * 4, 0x00020000);
  unsigned g_off = ((4 * wave + h) * N + min(n0 + j, N - 1)) * 4u, x_off = ((4 * wave + h) * K + min(k0 + j, K - 1)) * 4u;
  acc4 acc = 0.f;
  struct operands { float g[U], x[U]; };
  auto load = [&]() __attribute__((always_inline)) {
    operands o;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      o.g[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(gr, (int)g_off, 0, 0));
      o.x[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(xr, (int)x_off, 0, 0));
      g_off += 4 * W * 4u * N;
      x_off += 4 * W * 4u * K;
    }
    return o;
  };
  operands cur = load();
  for (int m0 = 4 * wave; m0 < M; m0 += 4 * W * U) {
    const operands nxt = load();
#pragma unroll
    for (int u = 0; u < U; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.g[u], cur.x[u], acc, 0, 0, 0);
    cur = nxt;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wave][r][lane] = acc[r];
  __syncthreads();
  if (wave >= 4) return;
  float s = red[0][wave][lane];  // wavefront r adds up register r
#pragma unroll
  for (int w = 1; w < W; ++w) s += red[w][wave][lane];
  const int n = n0 + 4 * h + wave, k = k0 + j;
  if (n < N && k < K) t.Y[(size_t)n * K + k] = s;
}

// How launch_weight_grads cuts a product: chunks of Y, groups of rows.
WeightGradTask plan_weight_grad(int M, int N, int K, int compute_units) {
  WeightGradTask p;
  p.M = M;
  p.N = N;
  p.K = K;
  // (some more tiles than compute units; 32-bit offsets, with a thousand rows past the end)
  p.few = M <= kWgFewRows && ((N + 15) / 16) * ((K + 15) / 16) <= 2 * compute_units && std::max(N, K) <= 16384;
  if (p.few) {
    p.n_chunks = (N + 15) / 16;
    p.k_chunks = (K + 15) / 16;
    return p;
  }
  // chunks of up to 64 columns of both, evenly (300 = 5 x 64, 128 = 2 x 64, 40 = 48)
  auto cut = [](int width, int &chunks, int &blocks) {
    chunks = (width + 63) / 64;
    blocks = std::min(width, ((width + chunks - 1) / chunks + 15) / 16);
    chunks = (width + 16 * blocks - 1) / (16 * blocks);
  };
  cut(N, p.n_chunks, p.nb);
  cut(K, p.k_chunks, p.kb);
  // eight wavefronts per compute unit, of a block of rows or more each
  // (a multiple of 8: the chunks of a block of rows on one XCD, whose L2 has the other operand and the lines two chunks share)
  const int chunks = p.n_chunks * p.k_chunks, blocks = (M + kWgRows - 1) / kWgRows;
  // Eight wavefronts a workgroup halve the sums that go through memory, where every wavefront of the device has a block of rows all the same (two groups
  // of four / one of eight, both launches: 100,000 rows 64 x 128 30.1 / 27.8 us, a layer 145 / 141; 131,072 rows 64 x 300 and 40 x 64 73 / 70, of a step of 280 that runs
  // differ by as much).
  p.waves = blocks >= 8 * compute_units ? 8 : 4;
  p.groups = std::max(1, std::min(std::max(1, 8 / p.waves * compute_units / chunks), (blocks + p.waves - 1) / p.waves));
  if (p.groups > 8) p.groups = p.groups / 8 * 8;
  return p;
}

// One gradient, or (second not null) two that share their launches where both are of few rows, or both are not.
hipError_t launch_weight_grads(const WeightGradTask &first, const WeightGradTask *second, hipStream_t st) {
  if (second && (second->few != first.few || second->waves != first.waves)) {
    const hipError_t err = launch_weight_grads(first, nullptr, st);
    return err != hipSuccess ? err : launch_weight_grads(*second, nullptr, st);
  }
  const WeightGradTask none;
  const WeightGradTask &b = second ? *second : none;
  const int first_blocks = first.blocks(), blocks = first_blocks + (second ? b.blocks() : 0);
  if (first.few) {
    hipLaunchKernelGGL(weight_grad_few_kernel, dim3(blocks), dim3(1024), 0, st, first, b, first_blocks);
    return hipGetLastError();
  }
  if (first.waves == 8) hipLaunchKernelGGL(weight_grad_kernel<8>, dim3(blocks), dim3(512), 0, st, first, b, first_blocks);
  else hipLaunchKernelGGL(weight_grad_kernel<4>, dim3(blocks), dim3(256), 0, st, first, b, first_blocks);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  auto registers = [](const WeightGradTask &t) { return t.nb * t.kb * 4 * t.n_chunks * t.k_chunks; };
  hipLaunchKernelGGL(weight_grad_reduce_kernel, dim3(registers(first) + (second ? registers(b) : 0)), dim3(256), 0, st, first, b, registers(first));
  return hipGetLastError();
}

}  // namespace tf
