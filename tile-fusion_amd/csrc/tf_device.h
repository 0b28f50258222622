// Device-side helpers shared by the kernel files of libtilefusion_hip (gfx950): the lane-group row
// products every sparse kernel is built from, vectors of floats, streaming loads and stores, the
// workgroup-to-XCD mapping and the LDS-only barrier.
#pragma once
#include <hip/hip_runtime.h>
#include <climits>
#include <cstdlib>

#include "tf_internal.h"

namespace tf {

#ifndef TF_BLOCK
#define TF_BLOCK 256
#endif
constexpr int kBlock = TF_BLOCK;  // threads per workgroup of the lane-group kernels
constexpr int kXcds = 8;     // workgroup ids are dealt round-robin over the 8 XCDs

template <int V> struct alignas(4 * V) fvec { float v[V]; };

template <int V> __device__ __forceinline__ fvec<V> vzero() {
  fvec<V> r;
#pragma unroll
  for (int i = 0; i < V; ++i) r.v[i] = 0.f;
  return r;
}
template <int V> __device__ __forceinline__ void vfma(float a, const fvec<V> &x, fvec<V> &acc) {
#pragma unroll
  for (int i = 0; i < V; ++i) acc.v[i] = __builtin_fmaf(a, x.v[i], acc.v[i]);
}
template <int V> __device__ __forceinline__ void vadd(const fvec<V> &x, fvec<V> &acc) {
#pragma unroll
  for (int i = 0; i < V; ++i) acc.v[i] += x.v[i];
}
// Output that this library does not read again leaves through a streaming (nontemporal) store.
template <int V> __device__ __forceinline__ void store_streaming(float *dst, const fvec<V> &v) {
  typedef float fv __attribute__((ext_vector_type(V)));
  fv x;
#pragma unroll
  for (int u = 0; u < V; ++u) x[u] = v.v[u];
  __builtin_nontemporal_store(x, reinterpret_cast<fv *>(dst));
}
template <> __device__ __forceinline__ void store_streaming<1>(float *dst, const fvec<1> &v) {
  __builtin_nontemporal_store(v.v[0], dst);
}
// ... and input that is read once, whole cache lines per instruction, comes through a streaming load.
__device__ __forceinline__ fvec<4> load_streaming4(const float *src) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  const f4 x = __builtin_nontemporal_load(reinterpret_cast<const f4 *>(src));
  fvec<4> r;
  r.v[0] = x[0]; r.v[1] = x[1]; r.v[2] = x[2]; r.v[3] = x[3];
  return r;
}

// A plain load of four floats as one value (assigning *(fvec<4> *) to a member of a struct in registers
// can stay a copy through private memory).
__device__ __forceinline__ fvec<4> load4(const float *src) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  const f4 x = *reinterpret_cast<const f4 *>(src);
  fvec<4> r;
  r.v[0] = x[0]; r.v[1] = x[1]; r.v[2] = x[2]; r.v[3] = x[3];
  return r;
}

// Consecutive workgroup ids land on different XCDs (each with its own 4 MB L2).  Work items
// are cut into chunks of `bpc` consecutive items and chunk c goes to XCD c % 8, so that an
// XCD walks whole chunks in order.  With bpc = all items / 8 every XCD gets one contiguous
// run (neighbouring tiles share halo rows in one L2); with bpc = (a far stencil stride) / 8
// every XCD keeps the same slab of every plane, so the plane above and below a row are
// still in its L2 when they are needed again.  bpc <= 0 switches the remapping off.
__device__ __forceinline__ int xcd_contiguous(int bid, int bpc) {
  if (bpc <= 0) return bid;
  const int xcd = bid % kXcds, s = bid / kXcds;
  return ((s / bpc) * kXcds + xcd) * bpc + (s % bpc);
}

// Work items per XCD for xcd_contiguous; 0 (identity mapping) when the environment variable
// TF_XCD_REMAP is set to 0.  The grid is sized grid_of(n) either way.
inline bool xcd_remap_on() {
  static const bool on = [] { const char *e = getenv("TF_XCD_REMAP"); return !(e && e[0] == '0'); }();
  return on;
}
inline int per_xcd_of(int n) { return xcd_remap_on() ? (n + kXcds - 1) / kXcds : 0; }
inline int grid_of(int n) { return (n + kXcds - 1) / kXcds * kXcds; }

// Workgroup barrier that orders LDS traffic only.  __syncthreads() also waits for every
// global load and store of the wavefront, which would cut off the loads a kernel issues
// ahead of time for a later phase; kernels that prefetch across barriers use this instead.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int V> struct GlobalRows {
  const float *__restrict__ base;
  int ld;    // row stride in floats
  int coff;  // this lane's first column
  __device__ __forceinline__ fvec<V> load(int row) const {
    return *reinterpret_cast<const fvec<V> *>(base + (size_t)row * ld + coff);
  }
};
template <int V> struct LdsRows {
  const float *base;  // slab; row r of the intermediate is at (r - first) * ld
  int ld, coff, first;
  __device__ __forceinline__ fvec<V> load(int row) const {
    return *reinterpret_cast<const fvec<V> *>(base + (row - first) * ld + coff);
  }
};

// acc += sum over stored entries k in [kb, ke) of val[k] * src.row(idx[k]), CSR order.
// All LPR lanes of the group must call this together (it shuffles inside the group).
// The group loads up to LPR (column, value) pairs with one coalesced load, then takes them
// eight (or four) at a time: all gathers of a batch are issued before its first fma, and a
// short last batch re-reads the last entry in its unused slots and skips their fma, so a
// short row costs one gather round trip instead of one per entry.
template <int V, int LPR, int B, class Src, bool FLAG = false>
__device__ __forceinline__ void row_dot_batch(int c, float a, int t, int cnt, bool col_ok, const Src &src,
                                              fvec<V> &acc) {
  int cc[B];
  float aa[B];
#pragma unroll
  for (int u = 0; u < B; ++u) {
    const int sl = min(t + u, cnt - 1);
    cc[u] = __shfl(c, sl, LPR);
    aa[u] = __shfl(a, sl, LPR);
  }
  if (col_ok) {
    fvec<V> x[B];
#pragma unroll
    for (int u = 0; u < B; ++u) {
      if constexpr (FLAG) x[u] = (t + u < cnt) ? src.load_flagged(cc[u]) : vzero<V>();
      else x[u] = (t + u < cnt) ? src.load(cc[u]) : vzero<V>();
    }
#pragma unroll
    for (int u = 0; u < B; ++u) {
      fvec<V> next = acc;
      vfma<V>(aa[u], x[u], next);
      if (t + u < cnt) acc = next;
    }
  }
}

// The same for cnt <= LPR entries already in registers: lane g of the group holds entry g.
template <int V, int LPR, class Src, bool FLAG = false>
__device__ __forceinline__ void row_dot_loaded(int c, float a, int cnt, bool col_ok, const Src &src,
                                               fvec<V> &acc) {
  int t = 0;
  if constexpr (LPR >= 8)
    for (; t + 8 <= cnt; t += 8) row_dot_batch<V, LPR, 8, Src, FLAG>(c, a, t, cnt, col_ok, src, acc);
  if (t + 4 <= cnt) { row_dot_batch<V, LPR, 4, Src, FLAG>(c, a, t, cnt, col_ok, src, acc); t += 4; }
  if (t < cnt) row_dot_batch<V, LPR, 4, Src, FLAG>(c, a, t, cnt, col_ok, src, acc);
}

template <int V, int LPR, class Src, bool FLAG = false>
__device__ __forceinline__ void row_dot(const int *__restrict__ idx, const float *__restrict__ val,
                                        int kb, int ke, int glane, bool col_ok, const Src &src,
                                        fvec<V> &acc) {
  for (int k0 = kb; k0 < ke; k0 += LPR) {
    const int k = k0 + glane;
    int c = 0;
    float a = 0.f;
    if (k < ke) { c = idx[k]; a = val[k]; }
    row_dot_loaded<V, LPR, Src, FLAG>(c, a, min(LPR, ke - k0), col_ok, src, acc);
  }
}

// The same sum with every lane reading the row's (column, value) pairs itself: the lanes of a
// group read the same address, which costs one request per group and no cross-lane traffic.
// Eight pairs, then their eight gathers, then the fmas; slots past the row's end load nothing.
// (Requesting the next eight pairs behind the current gathers, so that they arrive together, takes
// 112 registers instead of 60 and halves the wavefronts in flight: the R-MAT step went from 2.24 to
// 2.88 ms.  Wavefronts in flight are worth more to these launches than a shorter chain of dependent
// loads per row.)
template <int V, int LPR, class Src, bool FLAG = false>
__device__ __forceinline__ void row_dot_direct(const int *__restrict__ idx, const float *__restrict__ val,
                                               int kb, int ke, bool col_ok, const Src &src, fvec<V> &acc) {
  for (int k0 = kb; k0 < ke; k0 += 8) {
    int cc[8];
    float aa[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      cc[u] = 0;
      aa[u] = 0.f;
      if (k0 + u < ke) { cc[u] = idx[k0 + u]; aa[u] = val[k0 + u]; }
    }
    if (col_ok) {
      fvec<V> x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        if constexpr (FLAG) x[u] = (k0 + u < ke) ? src.load_flagged(cc[u]) : vzero<V>();
        else x[u] = (k0 + u < ke) ? src.load(cc[u]) : vzero<V>();
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        fvec<V> next = acc;
        vfma<V>(aa[u], x[u], next);
        if (k0 + u < ke) acc = next;
      }
    }
  }
}

// ---- dense products (tf_dense.hip, tf_rows.hip) ----
typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // (rows of K floats start at any multiple of 4 bytes)
typedef float acc4 __attribute__((ext_vector_type(4)));

// ---- fp32 products on the bf16 matrix cores ----
//
// A float is the sum of three bf16 of eight significant bits each, x = h + m + l, every difference exact: m is below 2^-8 of x, l below 2^-16.
// The product of two such sums without l l, below 2^-32 of it, is eight bf16 products, which v_mfma_f32_16x16x32_bf16 adds up in fp32 in
// 8 x 16 cycles per 32 values of k; v_mfma_f32_16x16x4_f32 takes 8 x 32.  (m l and l m reach 4.9e-8 of a product together: without them a row with one
// value that is not zero came out up to 1.1e-7 off where a rounded product is 6.0e-8 off.)  h h is added up in one accumulator and the seven small terms
// in another: the cores cut sums off instead of rounding them, and the large sum is then cut once per 32 values of k, and not at all
// while it has 24 bits.  Root mean square of the error over the sum of magnitudes, values in [-1, 1], K = 128, in e-8, for 1 / 2 / 4 / 8 / 128 values
// that are not zero: fp32 cores 2.53 / 2.54 / 2.53 / 2.48 / 2.40, this 2.53 / 2.09 / 1.64 / 1.26 / 0.70; largest of five million 6.0 / 11.3 / 17 / 22 / 30 and
// 6.0 / 15.0 / 14 / 15 / 9.
// bf16 has no bits below 2^-133 where floats end at 2^-149: both operands are made 2^20 times larger on the way in, which leaves every part of every float
// whole, and sums 2^-40 times smaller on the way out.  (Parts may be denormal: the cores take them as they are.  Operands of 2^-148 times 2^35 come out
// as precise as any others.)  Infinities, NaN, operands beyond 2^107 and sums beyond 2^87 come out infinite or NaN: the caller looks for those and
// computes such a block again on the fp32 cores.
// What the cores cut off when they align products is always cut downwards, some 4e-9 of a sum: nothing in one result, but 2e-7 in a
// weight gradient over 3,000 blocks of rows with as many terms of either sign.  Callers therefore scale rows of odd number, or every other block of them, by -2^20.
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
constexpr float kSplitIn = 0x1p20f, kSplitOut = 0x1p-40f;
template <class T> struct split3 { T h, m, l; };

// Two floats at a time, their parts read back out of the pair of bf16: 26 VALU instructions for four floats.  (Left to itself the compiler converts
// every value once for the pair and once for the difference: 34.  131,072 rows 300 x 64 34.2 -> 32.3 us, a weight gradient of 300 x 64 and 64 x 40
// over them 66.0 -> 56.6, 1,049,157 rows 128 x 128 219 -> 211, all in six products, together with the branch for K's last values in gemm_split_kernel.)
__device__ __forceinline__ void split2(float v0, float v1, float scale, unsigned &h, unsigned &m, unsigned &l) {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  typedef float f2 __attribute__((ext_vector_type(2)));
  const float x0 = v0 * scale, x1 = v1 * scale;
  h = __builtin_bit_cast(unsigned, __builtin_convertvector(f2{x0, x1}, bf2));
  const float r0 = x0 - __uint_as_float(h << 16), r1 = x1 - __uint_as_float(h & 0xffff0000u);
  m = __builtin_bit_cast(unsigned, __builtin_convertvector(f2{r0, r1}, bf2));
  l = __builtin_bit_cast(unsigned, __builtin_convertvector(f2{r0 - __uint_as_float(m << 16), r1 - __uint_as_float(m & 0xffff0000u)}, bf2));
}
__device__ __forceinline__ split3<bf4> split4(float v0, float v1, float v2, float v3, float scale = kSplitIn) {
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  unsigned h[2], m[2], l[2];
  split2(v0, v1, scale, h[0], m[0], l[0]);
  split2(v2, v3, scale, h[1], m[1], l[1]);
  return {__builtin_bit_cast(bf4, u2{h[0], h[1]}), __builtin_bit_cast(bf4, u2{m[0], m[1]}), __builtin_bit_cast(bf4, u2{l[0], l[1]})};
}
__device__ __forceinline__ split3<bf8> split8(const f4v &lo, const f4v &hi, float scale = kSplitIn) {
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  unsigned h[4], m[4], l[4];
  split2(lo[0], lo[1], scale, h[0], m[0], l[0]);
  split2(lo[2], lo[3], scale, h[1], m[1], l[1]);
  split2(hi[0], hi[1], scale, h[2], m[2], l[2]);
  split2(hi[2], hi[3], scale, h[3], m[3], l[3]);
  return {__builtin_bit_cast(bf8, u4{h[0], h[1], h[2], h[3]}), __builtin_bit_cast(bf8, u4{m[0], m[1], m[2], m[3]}), __builtin_bit_cast(bf8, u4{l[0], l[1], l[2], l[3]})};
}

// CB adjacent floats, at any multiple of four bytes.
template <int CB> struct cvec { float v[CB]; };

// The values v of CB adjacent columns at Y + at, the first `columns` of them existing ones.
template <int CB> __device__ __forceinline__ void gemm_store(float *__restrict__ Y, size_t at, cvec<CB> v, int columns, const GemmOut &how) {
  auto finish = [&](float x, size_t i) __attribute__((always_inline)) {
    if (how.accumulate) x += Y[i];
    if (how.mask) x = how.mask[i] <= 0.f ? 0.f : x;
    if (how.relu) x = x < 0.f ? 0.f : x;
    return x;
  };
  if (columns >= CB) {
    if (how.accumulate || how.mask || how.relu) {
      cvec<CB> m;
      if (how.mask) m = *reinterpret_cast<const cvec<CB> *>(how.mask + at);
      if (how.accumulate) {
        const cvec<CB> y = *reinterpret_cast<const cvec<CB> *>(Y + at);
#pragma unroll
        for (int c = 0; c < CB; ++c) v.v[c] += y.v[c];
      }
#pragma unroll
      for (int c = 0; c < CB; ++c) {
        if (how.mask) v.v[c] = m.v[c] <= 0.f ? 0.f : v.v[c];
        if (how.relu) v.v[c] = v.v[c] < 0.f ? 0.f : v.v[c];
      }
    }
    *reinterpret_cast<cvec<CB> *>(Y + at) = v;
  } else {
#pragma unroll
    for (int c = 0; c < CB; ++c)
      if (c < columns) Y[at + c] = finish(v.v[c], at + c);
  }
}
}  // namespace tf
