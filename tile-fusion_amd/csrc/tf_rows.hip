// Row-wise SpMM  Y[i,:] = sum_k Ax[k] * X[Ai[k],:]  for gfx950: the unfused remainder of a schedule (X = the
// intermediate in HBM), producer rows that no tile fuses, tf_spmm, and the reduction of long rows' partial sums.
// One lane group of LPR lanes owns one row, a lane V adjacent columns of it; the stored entries are walked in CSR
// order with one fma per element, as in the reference's AVX2 kernels
// (fusion/src/SpMM_SpMM_vectorized.cpp:892-936).  Small, short-lived workgroups: what hides the gather latency is
// the number of rows in flight.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <utility>

#include "tf_internal.h"
#include "tf_device.h"
#include "tf_rows.h"

namespace tf {

namespace {

// V floats at any multiple of four bytes: rows of N columns start anywhere when N is not a multiple of 4.
typedef float f4 __attribute__((ext_vector_type(4)));
template <int V> struct at4 { typedef float type __attribute__((ext_vector_type(V), aligned(4))); };
template <> struct at4<1> { typedef float type; };

template <int V> __device__ __forceinline__ fvec<V> load_any(const float *p) {
  fvec<V> r;
  const typename at4<V>::type x = *reinterpret_cast<const typename at4<V>::type *>(p);
  if constexpr (V == 1) r.v[0] = x;
  else {
#pragma unroll
    for (int u = 0; u < V; ++u) r.v[u] = x[u];
  }
  return r;
}
template <int V> __device__ __forceinline__ void store_any(float *p, const fvec<V> &v, bool streaming) {
  typename at4<V>::type x;
  if constexpr (V == 1) x = v.v[0];
  else {
#pragma unroll
    for (int u = 0; u < V; ++u) x[u] = v.v[u];
  }
  // (written out: the compiler makes one store of the two branches and drops the hint; the state that must pass before the registers of
  // sixteen bytes are written is then ours too)
  if (streaming && V == 4) asm volatile("global_store_dwordx4 %0, %1, off nt\n\ts_nop 0" ::"v"(p), "v"(x) : "memory");
  else if (streaming && V == 1) asm volatile("global_store_dword %0, %1, off nt" ::"v"(p), "v"(x) : "memory");
  else *reinterpret_cast<typename at4<V>::type *>(p) = x;
}

template <int V> struct RowsOf {
  const float *__restrict__ base;
  int ld;    // row stride in floats
  int coff;  // this lane's first column
  __device__ __forceinline__ fvec<V> load(int row) const { return load_any<V>(base + (size_t)row * ld + coff); }
  // A column index whose top bit is set names a row the schedule expects no second reader to find in L2
  // ("cold"): it is fetched with a streaming load, so that it does not push a row with readers out.
  __device__ __forceinline__ fvec<V> load_flagged(int c) const {
    const float *p = base + (size_t)(c & INT_MAX) * ld + coff;
    if (c < 0) {
      fvec<V> r;
      const typename at4<V>::type x = __builtin_nontemporal_load(reinterpret_cast<const typename at4<V>::type *>(p));
      if constexpr (V == 1) r.v[0] = x;
      else {
#pragma unroll
        for (int u = 0; u < V; ++u) r.v[u] = x[u];
      }
      return r;
    }
    return load_any<V>(p);
  }
};

// ---- the walk over a row's entries with the pairs handed round by DPP ----------------------------------
//
// Each lane loads one (column, value) pair of up to E = min(LPR, 16) consecutive entries (E = 4 for groups of 4 and 8 lanes),
// turns the column into the row's byte offset, and the other lanes of the group get both through a DPP broadcast that is
// the operand of the instruction that needs it: an entry costs one v_add_u32 (its gather's offset), one gather and four
// v_fmac_f32.  When every lane reads the pairs itself, the redundant copies are a third of what L1 returns, and every
// entry of a batch has a branch around its load.  Entries past a row's end take an offset past the end of X, for which a
// buffer load returns zeros without a memory access: no branches, and fma(0, 0, acc) leaves the sum as it is.  X may have up
// to 2 GB (32-bit offsets).
template <int E, int L> struct group_bcast;  // lane L of the 16 (E = 16), of the quad (E = 4), of the pair (E = 2)
#define TF_GROUP_BCAST(E_, CTRL)                                                                                       \
  template <int L> struct group_bcast<E_, L> {                                                                         \
    static __device__ __forceinline__ unsigned add(unsigned off, unsigned lane_off) {                                  \
      unsigned r;                                                                                                      \
      asm("s_nop 1\n\tv_add_u32_dpp %0, %1, %2 " CTRL(3) " row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(off), "v"(lane_off), "n"(L), "n"(L + 2)); \
      return r;                                                                                                        \
    }                                                                                                                  \
    static __device__ __forceinline__ void fma(float val, const f4 &x, fvec<4> &acc) {                                 \
      asm("s_nop 1\n\t"                                                                                                \
          "v_fmac_f32_dpp %0, %4, %5 " CTRL(9) " row_mask:0xf bank_mask:0xf\n\t"                                       \
          "v_fmac_f32_dpp %1, %4, %6 " CTRL(9) " row_mask:0xf bank_mask:0xf\n\t"                                       \
          "v_fmac_f32_dpp %2, %4, %7 " CTRL(9) " row_mask:0xf bank_mask:0xf\n\t"                                       \
          "v_fmac_f32_dpp %3, %4, %8 " CTRL(9) " row_mask:0xf bank_mask:0xf"                                           \
          : "+v"(acc.v[0]), "+v"(acc.v[1]), "+v"(acc.v[2]), "+v"(acc.v[3])                                             \
          : "v"(val), "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "n"(L), "n"(L + 2));                                 \
    }                                                                                                                  \
  }
#define TF_ROW16(N_) "row_newbcast:%" #N_
#define TF_QUAD(N_) "quad_perm:[%" #N_ ",%" #N_ ",%" #N_ ",%" #N_ "]"
TF_GROUP_BCAST(16, TF_ROW16);
TF_GROUP_BCAST(4, TF_QUAD);
#undef TF_GROUP_BCAST
// (a pair's other pair in the quad is another row's)
template <int L> struct group_bcast<2, L> {
  static __device__ __forceinline__ unsigned add(unsigned off, unsigned lane_off) {
    unsigned r;
    asm("s_nop 1\n\tv_add_u32_dpp %0, %1, %2 quad_perm:[%3,%3,%4,%4] row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(off), "v"(lane_off), "n"(L), "n"(L + 2));
    return r;
  }
  static __device__ __forceinline__ void fma(float val, const f4 &x, fvec<4> &acc) {
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %0, %4, %5 quad_perm:[%9,%9,%10,%10] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %4, %6 quad_perm:[%9,%9,%10,%10] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %2, %4, %7 quad_perm:[%9,%9,%10,%10] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %3, %4, %8 quad_perm:[%9,%9,%10,%10] row_mask:0xf bank_mask:0xf"
        : "+v"(acc.v[0]), "+v"(acc.v[1]), "+v"(acc.v[2]), "+v"(acc.v[3])
        : "v"(val), "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "n"(L), "n"(L + 2));
  }
};

__device__ __forceinline__ f4 buffer_gather(__amdgpu_buffer_rsrc_t x, unsigned off) {
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  const u4 v = __builtin_amdgcn_raw_buffer_load_b128(x, (int)off, 0, 0);
  return f4{__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3])};
}

// B entries, the pairs of entry u in lane (FIRST + u) % E of set (FIRST + u) / E.
template <int E, int FIRST, int B, int SETS>
__device__ __forceinline__ void dpp_batch(__amdgpu_buffer_rsrc_t X, const unsigned (&off)[SETS], const float (&val)[SETS], unsigned lane_off, fvec<4> &acc) {
  f4 x[B];
  [&]<int... U>(std::integer_sequence<int, U...>) __attribute__((always_inline)) {
    ((x[U] = buffer_gather(X, group_bcast<E, (FIRST + U) % E>::add(off[(FIRST + U) / E], lane_off))), ...);
    (group_bcast<E, (FIRST + U) % E>::fma(val[(FIRST + U) / E], x[U], acc), ...);
  }(std::make_integer_sequence<int, B>{});
}

template <int LPR>
__device__ __forceinline__ void row_dot_dpp(const int *__restrict__ idx, const float *__restrict__ val, int kb, int ke, int glane,
                                            __amdgpu_buffer_rsrc_t X, unsigned row_bytes, unsigned lane_off, fvec<4> &acc) {
  constexpr int E = LPR >= 16 ? 16 : LPR >= 4 ? 4 : 2, SETS = E == 16 ? 1 : 8 / E, STEP = E * SETS;
  const int mine = glane % E;
  for (int k0 = kb; k0 < ke; k0 += STEP) {
    unsigned off[SETS];
    float v[SETS];
#pragma unroll
    for (int s = 0; s < SETS; ++s) {
      const int k = k0 + s * E + mine;
      off[s] = 0x80000000u;
      v[s] = 0.f;
      if (k < ke) { off[s] = (unsigned)idx[k] * row_bytes; v[s] = val[k]; }
    }
    // (a branch of the wavefront: taken when some row of it has that many entries left)
    if (__ballot(ke - k0 > 4)) dpp_batch<E, 0, 8>(X, off, v, lane_off, acc);
    else dpp_batch<E, 0, 4>(X, off, v, lane_off, acc);
    if constexpr (STEP == 16) {
      if (__ballot(ke - k0 > 12)) dpp_batch<E, 8, 8>(X, off, v, lane_off, acc);
      else if (__ballot(ke - k0 > 8)) dpp_batch<E, 8, 4>(X, off, v, lane_off, acc);
    }
  }
}

template <int V> __device__ __forceinline__ void relu_of(fvec<V> &v) {
#pragma unroll
  for (int u = 0; u < V; ++u) v.v[u] = v.v[u] < 0.f ? 0.f : v.v[u];  // (a NaN stays one)
}

// Rows of Y without entries: the lane group of row q clears rows zero_rows[q], [q + n_rows], ... in the columns [c_begin, c_end),
// behind its own row, so that these stores wait for nothing and run beside the gathers.  (A launch of their own before the rows':
// 117 of 1,890 us on a 2^21-node R-MAT graph with 128 columns, 5 us each where it is four launches of a 2^17-node training step.)
// With accumulation there is something to do only for a ReLU, to what Y holds.
template <int V, int LPR>
__device__ __forceinline__ void clear_rows(const RowsArgs &a, int q, int glane, int c_begin, int c_end, int N, int accumulate) {
  for (int z = q; z < a.n_zero; z += a.n_rows) {
    float *y = a.Y + (size_t)a.zero_rows[z] * a.ldy;
    for (int c = c_begin + glane * V; c < c_end; c += LPR * V) {
      const int coff = V == 1 ? c : min(c, N - V);
      fvec<V> v = vzero<V>();
      if (accumulate) {
        v = load_any<V>(y + coff);
        relu_of<V>(v);
      }
      store_any<V>(y + coff, v, a.streaming);
    }
  }
}

}  // namespace

// ---------------------------------------------------------------------------------
// The workgroups of a launch: first chunk_blocks for the chunks of long rows (a workgroup each; a multiple of 8,
// those past n_chunks have nothing to do), so that the longest work starts first, then the rows.
//
// Chunks: the lane groups take eight entries of the chunk at a time, in turn, partial sums are combined inside a wavefront by shuffles
// and across the wavefronts through LDS, in a fixed order.  The only chunk of a row (slot < 0) goes straight to Y, a chunk of
// a row with several to partial[slot]; the last of a row's chunks to arrive adds them up in order (a launch of its own for that: 5 us
// after each of the four products of a training step of 345).  The last one sets
// the counter back to zero.
//
// Column slices (slices > 1): workgroup b works on the columns [4 LPR s, 4 LPR (s + 1)) of its rows with s = b mod 8 mod
// slices, so that an XCD gathers from one slice of X, `slices` times smaller than X; see slices_for.
//
// How a row's entries are walked: kDpp (above), the default; kDirect, every lane reads the pairs itself, for rows of fewer
// than four columns and for X beyond 2 GB; kMarked, the same with the schedule's "cold" mark in the columns' top bit.
//
// IN_PLACE: the values of listed rows are read where they are in the matrix' own array (RowsArgs::val_first).  A kernel of its own: with
// one for both a power-law step of kept values took 1,859 us instead of 1,847.
enum { kDirect, kMarked, kDpp };
template <int V, int LPR, int WALK, bool CHUNKS, bool IN_PLACE>
__global__ __launch_bounds__(kBlock) void spmm_rows_kernel(const RowsArgs a) {
  constexpr int G = kBlock / LPR;
  const int group = threadIdx.x / LPR, glane = threadIdx.x % LPR;
  __amdgpu_buffer_rsrc_t xr;
  if constexpr (WALK == kDpp) xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.X), 0, (int)(a.x_rows * a.ldx * 4u), 0x00020000);
  if constexpr (CHUNKS) {
    if (blockIdx.x < a.chunk_blocks) {
      if (blockIdx.x >= a.n_chunks) return;
      constexpr int kWaves = kBlock / 64, GW = 64 / LPR;  // lane groups of a wavefront
      __shared__ fvec<V> red[kWaves][LPR];
      const LongChunk ch = a.chunks[blockIdx.x];
      const int wave = threadIdx.x / 64;
      for (int c0 = 0; c0 < a.N; c0 += LPR * V) {
        const int col = c0 + glane * V;
        const bool ok = col < a.N;
        const int coff = clamp_col<V>(col, a.N);
        const RowsOf<V> src{a.X, a.ldx, coff};
        fvec<V> acc = vzero<V>();
        // (the direct walk: the other one beside it takes more than the 64 registers of eight wavefronts per SIMD)
        for (int k0 = ch.k_begin + group * 8; k0 < ch.k_end; k0 += G * 8)
          row_dot_direct<V, LPR>(a.chunk_Ai, a.chunk_Ax, k0, min(ch.k_end, k0 + 8), ok, src, acc);
        if constexpr (GW > 1) {
#pragma unroll
          for (int d = LPR; d < 64; d *= 2)
#pragma unroll
            for (int u = 0; u < V; ++u) acc.v[u] += __shfl_xor(acc.v[u], d, 64);
        }
        if (wave > 0 && threadIdx.x % 64 < LPR) red[wave][glane] = acc;
        __syncthreads();
        if (group == 0 && ok) {
#pragma unroll
          for (int w = 1; w < kWaves; ++w) vadd<V>(red[w][glane], acc);
          if (ch.slot < 0) {
            float *y = a.Y + (size_t)ch.row * a.ldy + coff;
            if (a.accumulate) vadd<V>(load_any<V>(y), acc);
            if (a.relu) relu_of<V>(acc);
            store_any<V>(y, acc, a.streaming);
          } else {
            float *p = a.partial + (size_t)ch.slot * a.N + coff;
#pragma unroll
            for (int u = 0; u < V; ++u) __hip_atomic_store(p + u, acc.v[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
        }
        __syncthreads();
      }
      if (ch.slot >= 0) {
        __shared__ int last;
        const LongRow lr = a.long_rows[a.chunk_long[blockIdx.x]];
        // (the sums are stored past this XCD's L2 and have to be there before the chunk counts as done; a fence would write back all of L2 and
        // made the launch 40 -> 74 us)
        if (wave == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (threadIdx.x == 0)
          last = __hip_atomic_fetch_add(a.arrived + a.chunk_long[blockIdx.x], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)lr.count - 1;
        __syncthreads();
        if (!last) return;
        if (threadIdx.x == 0) __hip_atomic_store(a.arrived + a.chunk_long[blockIdx.x], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (int c = threadIdx.x; c < a.N; c += kBlock) {
          float *y = a.Y + (size_t)lr.row * a.ldy + c;
          float s = a.accumulate ? *y : 0.f;
          for (int p = 0; p < lr.count; ++p) s += __hip_atomic_load(a.partial + (size_t)(lr.first + p) * a.N + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          *y = a.relu && s < 0.f ? 0.f : s;
        }
      }
      return;
    }
  }
  // The workgroups live for a microsecond or two: the arguments are all requested at once here, not one after the other
  // where they are first used, and a listed row's place in Y is not waited for before its entries are.
  asm volatile("" ::"s"(a.rows), "s"(a.Ap), "s"(a.Ai), "s"(a.Ax), "s"(a.X), "s"(a.Y), "s"(a.ldx), "s"(a.ldy), "s"(a.N), "s"(a.n_rows),
               "s"(a.accumulate), "s"(a.streaming), "s"(a.compact), "s"(a.relu), "s"(a.n_blocks), "s"(a.per_xcd), "s"(a.slices), "s"(a.n_zero));
  int b = CHUNKS ? blockIdx.x - a.chunk_blocks : blockIdx.x, c_begin = 0, c_end = a.N;
  if (a.slices > 1) {
    const int xcd = b % kXcds;
    b = b / kXcds * (kXcds / a.slices) + xcd / a.slices;
    c_begin = xcd % a.slices * (LPR * V);
    c_end = min(a.N, c_begin + LPR * V);
  } else {
    b = xcd_contiguous(b, a.per_xcd);
  }
  if (b >= a.n_blocks) return;
  const int q = b * G + group;
  if (q >= a.n_rows) return;  // whole lane groups leave together
  // compact: the CSR arrays hold the listed rows only, in the order of the list (the reference's
  // reordered adjacency: consumer rows stored in schedule order), so row q of them is row rows[q] of Y
  int r = q, i = q;
  if (a.rows) {
    i = a.rows[q];
    if (!a.compact) r = i;
  }
  const int kb = a.Ap[r], ke = a.Ap[r + 1];
  const float *ax = a.Ax;
  if constexpr (IN_PLACE) ax += a.val_first[q] - kb;
  for (int c0 = c_begin; c0 < c_end; c0 += LPR * V) {
    const int col = c0 + glane * V;
    const bool ok = col < a.N;
    const int coff = clamp_col<V>(col, a.N);
    const RowsOf<V> src{a.X, a.ldx, coff};
    float *y = a.Y + (size_t)i * a.ldy + coff;
    fvec<V> acc = vzero<V>();
    if (a.accumulate && ok) acc = load_any<V>(y);
    if constexpr (WALK == kDpp) row_dot_dpp<LPR>(a.Ai, ax, kb, ke, glane, xr, a.ldx * 4u, coff * 4u, acc);
    else row_dot_direct<V, LPR, RowsOf<V>, WALK == kMarked>(a.Ai, ax, kb, ke, ok, src, acc);
    if (ok) {
      if (a.relu) relu_of<V>(acc);
      store_any<V>(y, acc, a.streaming);
    }
  }
  if (a.n_zero > 0) clear_rows<V, LPR>(a, q, glane, c_begin, c_end, a.N, a.accumulate);
}

// ---------------------------------------------------------------------------------
// The same for rows whose columns rise and are spread over an X that no L2 holds: all rows in flight read the same stretch of X at the
// same time.  A lane group owns kSweepRows rows and takes at most one entry of each per step, if its column lies in front of a
// limit that rises with the steps; every XCD's workgroups (of one column slice where there are slices) start together and take steps of the same
// length, so that more of an XCD's gathers hit what another row has just fetched.  Bound: the lines that come from the Infinity Cache once
// per XCD and generation of workgroups, then L2 (100,000 rows of 11, N = 128: 67 us, 563 MB gathered; 77.5 in spmm_rows_kernel).  Nothing depends on the timing but time: entries are added in the row's order.
// Four rows a group are what 64 registers hold, of eight wavefronts per SIMD; eight rows and half the wavefronts read the same at N = 64 (36.1 / 34.2 us)
// and 4 % faster at 128.  Each lane group keeps kSweepEntries entries of each row in LDS, behind them a mark that lies in front of no limit, and refills when its
// wavefront has used all of them up.
// ---------------------------------------------------------------------------------
constexpr unsigned kSweepEnd = 0xffffffffu;
template <int LPR>
__global__ __launch_bounds__(kBlock, LPR == 4 ? 4 : 8) void sweep_rows_kernel(const RowsArgs a) {
  constexpr int G = kBlock / LPR, R = kSweepRows, E = kSweepEntries;
  __shared__ uint2 pairs[G][R][E + 1];  // byte offset in X and value
  const int group = threadIdx.x / LPR, glane = threadIdx.x % LPR;
  asm volatile("" ::"s"(a.Ap), "s"(a.Ai), "s"(a.Ax), "s"(a.X), "s"(a.Y), "s"(a.ldx), "s"(a.ldy), "s"(a.N), "s"(a.n_rows), "s"(a.accumulate),
               "s"(a.streaming), "s"(a.relu), "s"(a.slices), "s"(a.sweep_steps), "s"(a.sweep_bytes));
  const int xcd = blockIdx.x % kXcds, b = blockIdx.x / kXcds * (kXcds / a.slices) + xcd / a.slices;
  const int c_begin = xcd % a.slices * (LPR * 4);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.X), 0, (int)(a.x_rows * a.ldx * 4u), 0x00020000);
  const int q0 = (b * G + group) * R, n = min(max(a.n_rows - q0, 0), R);  // (a group without rows stays with its wavefront)
  const int col = c_begin + glane * 4, coff = clamp_col<4>(col, a.N);
  const bool ok = col < a.N;
  int at[R + 1];  // the rows' next entries to go to LDS, and their end
#pragma unroll
  for (int r = 0; r <= R; ++r) at[r] = n > 0 ? a.Ap[q0 + min(r, n)] : 0;
  int len[R];
#pragma unroll
  for (int r = 0; r < R; ++r) len[r] = at[r + 1] - at[r];
  fvec<4> acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    acc[r] = vzero<4>();
    if (a.accumulate && ok && r < n) acc[r] = load_any<4>(a.Y + (size_t)(q0 + r) * a.ldy + coff);
  }
  unsigned limit = a.sweep_bytes;
  int steps = a.sweep_steps;
  for (;;) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int k0 = 0; k0 <= E; k0 += LPR) {
        const int k = k0 + glane;
        uint2 e = {kSweepEnd, 0u};
        if (k < E && k < len[r]) {
          e.x = (unsigned)a.Ai[at[r] + k] * (a.ldx * 4u);
          e.y = __float_as_uint(a.Ax[at[r] + k]);
        }
        if (k <= E) pairs[group][r][k] = e;
      }
    // (a lane group reads what its own lanes have written: of one wavefront, in order)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    int k[R];
#pragma unroll
    for (int r = 0; r < R; ++r) k[r] = 0;
    for (;;) {
      f4 x[R];
      float v[R];
      bool left = false;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint2 e = pairs[group][r][k[r]];
        const bool take = e.x < limit;  // (never the mark)
        left |= e.x != kSweepEnd;
        x[r] = buffer_gather(xr, take ? e.x + coff * 4u : 0x80000000u);  // (past the end of X: zeros, without a memory access)
        v[r] = take ? __uint_as_float(e.y) : 0.f;
        k[r] += take;
      }
      if (!__ballot(left)) break;
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[r].v[u] = __builtin_fmaf(v[r], x[r][u], acc[r].v[u]);
      limit = --steps > 0 ? limit + a.sweep_bytes : kSweepEnd;
    }
    bool more = false;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      at[r] += E;
      len[r] -= E;
      more |= len[r] > 0;
    }
    if (!__ballot(more)) break;
    __builtin_amdgcn_wave_barrier();
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r < n && ok) {
      if (a.relu) relu_of<4>(acc[r]);
      store_any<4>(a.Y + (size_t)(q0 + r) * a.ldy + coff, acc[r], a.streaming);
    }
  }
}

// ---------------------------------------------------------------------------------
// Y = (A X) W in one launch: the rows of A X, K columns wide, are gathered as in spmm_rows_kernel into LDS, R of them a
// workgroup, and multiplied by W (K x N, or N x K with WT) on v_mfma_f32_16x16x4_f32; neither intermediate nor second
// launch.  In the product a wavefront owns 16 rows and 16 V columns (column V j + v of its panel is column block v's lane j).
// R = 16, for few rows: what counts is the chain of dependent loads, so the four wavefronts share the columns and W's first
// four steps are requested before the gathers.  R = 64, for many rows of up to 32 columns of X: what counts is L2, so W is
// read once per 64 rows and seven workgroups share a compute unit, one gathering while another multiplies.  See
// one_launch in tf_api.cpp for where this is the faster way.
// ---------------------------------------------------------------------------------
template <int LPR, int R, int V, bool WT, bool IN_PLACE>
__global__ __launch_bounds__(kBlock, R == 16 ? 1 : 7) void spmm_gemm_kernel(const RowsArgs a, const float *__restrict__ W, int N, const GemmOut how) {
  extern __shared__ __align__(16) float slab[];
  constexpr int G = kBlock / LPR, RT = R / 16, CW = 4 / RT;  // lane groups; row tiles; wavefronts side by side in columns
  const int K = a.N, ld = (K + 15) / 16 * 16 + 4;            // (four floats behind a row: its reads start in other banks)
  const int group = threadIdx.x / LPR, glane = threadIdx.x % LPR;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.X), 0, (int)(a.x_rows * a.ldx * 4u), 0x00020000);
  const int block = xcd_contiguous(blockIdx.x, a.per_xcd);
  if (block >= a.n_blocks) return;
  const int q0 = block * R;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, j = lane % 16, h = lane / 16;
  const int rt = wave % RT, S = (K + 15) / 16, full = K / 16;
  const int first_col = wave / RT * 16 * V + V * j;
  const float *sp = slab + (rt * 16 + j) * ld + 4 * h;
  struct panel { f4v b[V]; };
  // step s of W for this lane's columns (32-bit offsets: W is far smaller than 4 GB)
  auto load = [&](int col0, int s) __attribute__((always_inline)) {
    panel o;
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const unsigned c = min(col0 + v, N - 1), k0 = 16 * s + 4 * h;
      if (s < full) {
        if constexpr (WT) o.b[v] = *reinterpret_cast<const f4u *>(W + (c * (unsigned)K + k0));
        else {
#pragma unroll
          for (int t = 0; t < 4; ++t) o.b[v][t] = W[(k0 + t) * (unsigned)N + c];
        }
      } else {  // values of k past K
#pragma unroll
        for (int t = 0; t < 4; ++t) o.b[v][t] = k0 + t < (unsigned)K ? W[WT ? c * (unsigned)K + k0 + t : (k0 + t) * (unsigned)N + c] : 0.f;
      }
    }
    return o;
  };
  constexpr int AHEAD = R == 16 ? 4 : 1;  // steps of W requested ahead
  panel w[AHEAD];
  if (R == 16 && first_col < N) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) w[u] = load(first_col, min(u, S - 1));
  }
  for (int r = group; r < R; r += G) {
    const int q = q0 + r;
    int kb = 0, ke = 0;
    const float *ax = a.Ax;
    if (q < a.n_rows) {
      const int row = a.rows && !a.compact ? a.rows[q] : q;
      kb = a.Ap[row];
      ke = a.Ap[row + 1];
      if constexpr (IN_PLACE) ax += a.val_first[q] - kb;
    }
    for (int c0 = 0; c0 < K; c0 += LPR * 4) {
      const int col = c0 + glane * 4, coff = clamp_col<4>(col, K);
      fvec<4> acc = vzero<4>();
      row_dot_dpp<LPR>(a.Ai, ax, kb, ke, glane, xr, a.ldx * 4u, coff * 4u, acc);
      if (col < K) {
        float *s = slab + r * ld + coff;
        if (K % 4 == 0) *reinterpret_cast<fvec<4> *>(s) = acc;
        else { s[0] = acc.v[0]; s[1] = acc.v[1]; s[2] = acc.v[2]; s[3] = acc.v[3]; }
      }
    }
    if (glane < ld - 4 - K) slab[r * ld + K + glane] = 0.f;  // (up to 15 columns that fill the last step of k)
    if (LPR < 16)
      for (int c = glane + LPR; c < ld - 4 - K; c += LPR) slab[r * ld + K + c] = 0.f;
  }
  __syncthreads();
  for (int col0 = first_col; col0 - V * j < N; col0 += CW * 16 * V) {
    acc4 acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = 0.f;
    if (R != 16 || col0 != first_col) {
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) w[u] = load(col0, min(u, S - 1));
    }
    for (int s0 = 0; s0 < S; s0 += AHEAD) {
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        const int s = s0 + u;
        if (s >= S) break;
        const panel cur = w[u];
        if (s + AHEAD < S) w[u] = load(col0, s + AHEAD);
        const f4v x = *reinterpret_cast<const f4v *>(sp + 16 * s);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int v = 0; v < V; ++v) acc[v] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[t], cur.b[v][t], acc[v], 0, 0, 0);
      }
    }
    if (col0 < N) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int q = q0 + rt * 16 + 4 * h + r;
        if (q >= a.n_rows) continue;
        cvec<V> out;
#pragma unroll
        for (int v = 0; v < V; ++v) out.v[v] = acc[v][r];
        gemm_store<V>(a.Y, (size_t)(a.rows ? a.rows[q] : q) * a.ldy + col0, out, N - col0, how);
      }
    }
  }
  if (a.n_zero > 0) {
    for (int r = group; r < R && q0 + r < a.n_rows; r += G) {
      if (N >= 4) clear_rows<4, LPR>(a, q0 + r, glane, 0, N, N, how.accumulate);
      else clear_rows<1, LPR>(a, q0 + r, glane, 0, N, N, how.accumulate);
    }
  }
}

// Y[row] (+)= the sums in partial[seg_of[first .. first + count)] of the long rows' segments, in order.  The rows from n_big on have a
// lane group each, every lane four adjacent columns, the partial rows of eight segments requested before the first is added.
// The first n_big rows have groups of segments (slots from n_seg on name them): a workgroup each, a group of segments per lane
// group at a time, the groups' sums added in order through LDS.  (The groups in a launch before the rows': 37 us for both on a
// 2^18-node R-MAT graph, N = 128; 25 us in one.)
constexpr int kSegBlock = kBlock;
template <int V, int LPR>
__global__ __launch_bounds__(kSegBlock) void long_seg_reduce_kernel(const LongRow *__restrict__ rows, int n_long, int n_big,
                                                                    const LongRow *__restrict__ groups, int n_seg,
                                                                    const int *__restrict__ seg_of, const float *__restrict__ partial,
                                                                    float *__restrict__ Y, int ldy, int N, int accumulate, int relu) {
  constexpr int G = kSegBlock / LPR;
  __shared__ fvec<V> red[G][LPR];
  const int group = threadIdx.x / LPR, glane = threadIdx.x % LPR;
  auto add_up = [&](int first, int count, int coff, fvec<V> &acc) __attribute__((always_inline)) {
    for (int p0 = 0; p0 < count; p0 += 8) {
      fvec<V> x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (p0 + u < count) x[u] = load_any<V>(partial + (size_t)seg_of[first + p0 + u] * N + coff);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (p0 + u < count) vadd<V>(x[u], acc);
    }
  };
  const bool big = (int)blockIdx.x < n_big;
  const int q = big ? blockIdx.x : n_big + (blockIdx.x - n_big) * G + group;
  if (q >= n_long) return;
  const LongRow lr = rows[q];
  const int g_first = big ? seg_of[lr.first] - n_seg : 0;
  for (int c0 = 0; c0 < N; c0 += LPR * V) {
    const bool ok = c0 + glane * V < N;
    const int coff = clamp_col<V>(c0 + glane * V, N);
    float *y = Y + (size_t)lr.row * ldy + coff;
    fvec<V> acc = vzero<V>();
    if (big) {
      if (accumulate && group == 0 && ok) acc = load_any<V>(y);
      for (int g0 = 0; g0 < lr.count; g0 += G) {
        fvec<V> s = vzero<V>();
        if (g0 + group < lr.count) {
          const LongRow g = groups[g_first + g0 + group];
          add_up(g.first, g.count, coff, s);
        }
        red[group][glane] = s;
        __syncthreads();
        if (group == 0)
          for (int t = 0; t < G && g0 + t < lr.count; ++t) vadd<V>(red[t][glane], acc);
        __syncthreads();
      }
      if (group > 0 || !ok) continue;
    } else {
      if (!ok) continue;
      if (accumulate) acc = load_any<V>(y);
      add_up(lr.first, lr.count, coff, acc);
    }
    if (relu) relu_of<V>(acc);
    store_any<V>(y, acc, false);
  }
}

// ---- launchers ----------------------------------------------------------------------

namespace {

// How a.n_blocks workgroups of `rows` rows are dealt to the XCDs -- 0: workgroup b takes block b; > 0: chunks of rows per XCD turn;
// < 0: one contiguous run per XCD -- and the workgroups to launch for it.
int deal_to_xcds(RowsArgs &a, int xcd_chunk_rows, int rows) {
  const int n = a.n_blocks, want = xcd_chunk_rows > 0 ? std::max(1, xcd_chunk_rows / rows) : 0;
  a.per_xcd = xcd_chunk_rows == 0 || !xcd_remap_on() ? 0 : (want <= 0 || want * kXcds >= n) ? (n + kXcds - 1) / kXcds : want;
  const int per = std::max(a.per_xcd, 1) * kXcds;
  return (n + per - 1) / per * per;
}

#define TF_DISPATCH_ROWS(S_, CALL)                                              \
  do {                                                                          \
    if (S_.V == 1) { if (S_.LPR == 4) { CALL(1, 4); } else { CALL(1, 64); } }   \
    else if (S_.LPR == 2) { CALL(4, 2); } else if (S_.LPR == 4) { CALL(4, 4); } \
    else if (S_.LPR == 8) { CALL(4, 8); } else if (S_.LPR == 16) { CALL(4, 16); } \
    else if (S_.LPR == 32) { CALL(4, 32); } else { CALL(4, 64); }               \
  } while (0)

}  // namespace

hipError_t launch_spmm_rows(RowsArgs a, const RowsHow &how, hipStream_t st) {

  if (a.n_rows <= 0 && a.n_chunks <= 0) return hipSuccess;
  RowShape s = row_shape(a.N, a.accumulate);
  a.chunk_blocks = (a.n_chunks + kXcds - 1) / kXcds * kXcds;
  a.slices = s.V == 4 && !how.flagged && how.xcd_chunk_rows == 0 ? slices_for(a) : 1;
  if (a.slices > 1) s.LPR = kSliceCols / 4;
  const SweepShape sweep = sweep_for(a, how);
  if (sweep.LPR > 0) {
    const int rows = kBlock / sweep.LPR * kSweepRows, per = kXcds / sweep.slices;
    a.slices = sweep.slices;
    a.n_blocks = (a.n_rows + rows - 1) / rows;
    a.sweep_steps = sweep.steps;
    a.sweep_bytes = (unsigned)((unsigned long long)a.x_rows * a.ldx * 4 / sweep.steps + 1);
    const dim3 grid((a.n_blocks + per - 1) / per * kXcds);
#define CALLS(L_) hipLaunchKernelGGL((sweep_rows_kernel<L_>), grid, dim3(kBlock), 0, st, a)
    if (sweep.LPR == 4) CALLS(4); else if (sweep.LPR == 8) CALLS(8); else if (sweep.LPR == 16) CALLS(16); else CALLS(32);
#undef CALLS
    return hipGetLastError();
  }
  const int G = kBlock / s.LPR;
  a.n_blocks = (std::max(a.n_rows, 0) + G - 1) / G;
  const int blocks = deal_to_xcds(a, how.xcd_chunk_rows, G);
  const int turns = kXcds / a.slices;  // row blocks per eight workgroups
  const dim3 grid(a.chunk_blocks + (a.slices > 1 ? (a.n_blocks + turns - 1) / turns * kXcds : blocks));
#define CALL4(V_, L_, WALK_, CH_, IN_) hipLaunchKernelGGL((spmm_rows_kernel<V_, L_, WALK_, CH_, IN_>), grid, dim3(kBlock), 0, st, a)
#define CALL3(V_, L_, WALK_, CH_) do { if (a.val_first) { CALL4(V_, L_, WALK_, CH_, true); } else { CALL4(V_, L_, WALK_, CH_, false); } } while (0)
#define CALL2(V_, L_, WALK_) do { if (a.n_chunks > 0) { CALL3(V_, L_, WALK_, true); } else { CALL3(V_, L_, WALK_, false); } } while (0)
#define CALLP(V_, L_) do { if constexpr (V_ == 4) { CALL2(V_, L_, kDpp); } } while (0)
#define CALLD(V_, L_) CALL2(V_, L_, kDirect)
#define CALLM(V_, L_) CALL2(V_, L_, kMarked)
  // The DPP walk pays where L1 or L2 serves the gathers (27 points, 80^3, N = 64: 154 -> 116 us; R-MAT 2^20, N = 32: 311 -> 284)
  // and costs a little where the Infinity Cache does, rows in no order and X beyond 48 MB (Erdos-Renyi, 200,000 rows,
  // N = 64 / 100: 85.2 -> 87.0, 159.5 -> 162.3).
  const unsigned long long x_bytes = (unsigned long long)a.x_rows * a.ldx * 4;
  const bool far_gathers = a.compact && a.N >= 64 && x_bytes > (48ull << 20);
  if (how.flagged) TF_DISPATCH_ROWS(s, CALLM);
  else if (s.V == 4 && x_bytes <= 0x80000000ull && !far_gathers) TF_DISPATCH_ROWS(s, CALLP);
  else TF_DISPATCH_ROWS(s, CALLD);
#undef CALLP
#undef CALLD
#undef CALLM
#undef CALL2
#undef CALL3
#undef CALL4
  return hipGetLastError();
}

// Y = (A X) W for the rows of `a` (a.N = K the columns of X, a.ldy that of Y): K and N as spmm_gemm_fits says, X of up to 2 GB, no
// long rows.
hipError_t launch_spmm_gemm(RowsArgs a, const RowsHow &rows, const float *W, int wt, int N, const GemmOut &how, hipStream_t st) {
  if (a.n_rows <= 0) return hipSuccess;
  if (!spmm_gemm_fits(a.n_rows, a.N, N) || a.n_chunks > 0 || (unsigned long long)a.x_rows * a.ldx * 4 > 0x80000000ull) return hipErrorInvalidValue;
  const RowShape s = row_shape(a.N, 0);
  const int R = spmm_gemm_rows(a.n_rows), lds = (int)spmm_gemm_lds(a.n_rows, a.N);
  a.n_blocks = (a.n_rows + R - 1) / R;
  const dim3 grid(deal_to_xcds(a, rows.xcd_chunk_rows, R));
  hipError_t err = hipSuccess;
#define CALL4(L_, R_, V_, WT_, IN_)                                                                                                    \
  do {                                                                                                                                 \
    if (lds > 65536)                                                                                                                   \
      err = hipFuncSetAttribute(reinterpret_cast<const void *>(spmm_gemm_kernel<L_, R_, V_, WT_, IN_>), hipFuncAttributeMaxDynamicSharedMemorySize, lds); \
    if (err == hipSuccess) hipLaunchKernelGGL((spmm_gemm_kernel<L_, R_, V_, WT_, IN_>), grid, dim3(kBlock), lds, st, a, W, N, how);    \
  } while (0)
#define CALL3(L_, R_, V_, WT_) do { if (a.val_first) { CALL4(L_, R_, V_, WT_, true); } else { CALL4(L_, R_, V_, WT_, false); } } while (0)
#define CALL2(L_, R_, V_) do { if (wt) { CALL3(L_, R_, V_, true); } else { CALL3(L_, R_, V_, false); } } while (0)
#define CALL(V__, L_)                                                                                                   \
  do {                                                                                                                  \
    if constexpr (V__ == 4) {                                                                                           \
      if (R == 16) { if (N > 64) { CALL2(L_, 16, 2); } else { CALL2(L_, 16, 1); } } else if (N > 16) { CALL2(L_, 64, 2); } else { CALL2(L_, 64, 1); } \
    }                                                                                                                   \
  } while (0)
  TF_DISPATCH_ROWS(s, CALL);
#undef CALL
#undef CALL2
#undef CALL3
#undef CALL4
  return err != hipSuccess ? err : hipGetLastError();
}

// The long rows' sums of their segments' partial sums; the rows with groups of segments come first.
hipError_t launch_seg_reduce(const LongRow *rows, int n_rows, int n_big, const LongRow *groups, int n_seg, const int *seg_of, const float *partial,
                             float *Y, int ldy, int N, int accumulate, int relu, hipStream_t st) {
  if (n_rows <= 0) return hipSuccess;
  const RowShape s = row_shape(N, accumulate);
  const int G = kSegBlock / s.LPR;
#define CALL(V_, L_)                                                                                                                       \
  hipLaunchKernelGGL((long_seg_reduce_kernel<V_, L_>), dim3(n_big + (n_rows - n_big + G - 1) / G), dim3(kSegBlock), 0, st, rows, n_rows, n_big, \
                     groups, n_seg, seg_of, partial, Y, ldy, N, accumulate, relu)
  TF_DISPATCH_ROWS(s, CALL);
#undef CALL
  return hipGetLastError();
}

}  // namespace tf
