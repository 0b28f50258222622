// Fused SpMM-SpMM on the 27-point stencil of a 3D grid (gfx950): D = A (B C), A and B the pattern in which every grid point reads
// all its neighbours within one step in every direction, x fastest (checked against the matrices by the inspector: build_box in
// tf_march.cpp).  Any values.  The reference's answer to such patterns is tiling with redundancy (fusion/src/SpMM_SpMM.cpp:984-1057).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <utility>

#include "tf_internal.h"
#include "tf_device.h"

namespace tf {

namespace {

constexpr unsigned kNowhere = 0x80000000u;  // past the end of every buffer: loads give zeros

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

__device__ __forceinline__ float lds_read(unsigned addr) { return *reinterpret_cast<const __attribute__((address_space(3))) float *>(addr); }
__device__ __forceinline__ void lds_write(unsigned addr, float v) { *reinterpret_cast<__attribute__((address_space(3))) float *>(addr) = v; }

// One axis of the pattern: the entries a point has along it, and those of the points before it.
__device__ __forceinline__ int axis_count(int i, int n) { return 1 + (i > 0) + (i < n - 1); }
__device__ __forceinline__ int axis_before(int i) { return max(3 * i - 1, 0); }

// The values with which plane z of C (or of the intermediate) goes into the rows of the points (x + q, y), q < Q: of the rows in planes z - 1, z and
// z + 1 their last, middle and first nine.  A plane's rows are loaded once, lane 9 q + j taking values j, 9 + j and 18 + j of a row, and the middle and the
// last ones kept until their planes come.  They go through LDS to the lanes in which a broadcast of the matrix cores wants them: value j of
// plane z - 1 + i in lane 4 j + i, a register a point.
template <int Q> struct BoxValues {
  static constexpr int kBytes = 3 * 9 * Q * 4;  // of LDS, a wavefront
  __amdgpu_buffer_rsrc_t from;
  int x, y, nx, ny, nz, plane;  // plane: values of a line pair of axes, (3 nx - 2) (3 ny - 2)
  unsigned k[3];                // bytes, for plane 1 of many
  float next[3], middle, last[2];
  __device__ __forceinline__ void init(const float *values, unsigned bytes, int x_, int y_, const BoxArgs &a, int lane, bool any) {
    from = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(values), 0, (int)bytes, 0x00020000);
    x = x_; y = y_; nx = a.nx; ny = a.ny; nz = a.nz;
    plane = (3 * nx - 2) * (3 * ny - 2);
    const int j = lane % 9, jy = j / 3, jx = j % 3, xq = x + lane / 9;
    const int cx = axis_count(xq, nx), cy = axis_count(y, ny), row = axis_before(y) * (3 * nx - 2) + cy * axis_before(xq);
    const bool there = any && lane < 9 * Q && xq >= 0 && xq < nx && y >= 0 && y < ny && xq + jx >= 1 && xq + jx <= nx && y + jy >= 1 && y + jy <= ny;
#pragma unroll
    for (int b = 0; b < 3; ++b) k[b] = there ? 4u * (unsigned)(2 * plane + 3 * row + (b * cy + jy - (y == 0)) * cx + jx - (xq == 0)) : kNowhere;
  }
  // asks for the rows in plane z
  __device__ __forceinline__ void load(int z, int lane) {
    unsigned at[3] = {k[0], k[1], k[2]};
    int so = 0;
    if (z >= 1 && z <= nz - 2) {
      so = (z - 1) * 12 * plane;
    } else {  // shorter rows, or none
      int xq = x + lane / 9, ys = y;
      asm volatile("" : "+v"(xq), "+s"(ys));  // (what follows is made here: kept over the loop it takes registers)
      const int cy = axis_count(ys, ny), row = axis_before(ys) * (3 * nx - 2) + cy * axis_before(xq), nine = cy * axis_count(xq, nx);
      const unsigned less = 4u * (unsigned)(z == 0 ? 2 * plane + row + nine : row);
      if (z > 0) so = (nz - 2) * 12 * plane;
#pragma unroll
      for (int b = 0; b < 3; ++b) at[b] = z < 0 || z >= nz || (z == 0 && b == 0) || (z == nz - 1 && b == 2) || k[b] >= kNowhere ? kNowhere : k[b] - less;
    }
#pragma unroll
    for (int b = 0; b < 3; ++b) next[b] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(from, (int)at[b], so, 0));
  }
  // what was asked for is there: the next plane's values to LDS
  __device__ __forceinline__ void put(unsigned to, int lane) {
    if (lane < 9 * Q) {
      lds_write(to + lane * 4, last[1]);
      lds_write(to + 36 * Q + lane * 4, middle);
      lds_write(to + 72 * Q + lane * 4, next[0]);
    }
    turn();
  }
  __device__ __forceinline__ void turn() {
    last[1] = last[0];
    last[0] = next[2];
    middle = next[1];
  }
  // (lanes that name no value take some other one: their products are in rows nobody reads)
  static __device__ __forceinline__ unsigned place(unsigned at, int lane) { return at + min(lane % 4, 2) * 36 * Q + min(lane / 4, 8) * 4; }
};

}  // namespace

// A run is a column of 2 Q x by grid points and a range of planes, 64 columns of C wide; a workgroup walks it plane by plane, a wavefront with Q + 1
// points of a line of the intermediate (the column and one point around it) and Q of D, a lane with one column.  Step z:
//   plane z + 1 of C comes into LDS, and of both matrices the next rows' values;
//   plane z of C goes into the rows of the intermediate in planes z - 1, z and z + 1, whose sums are in registers; plane z - 1 is whole then, and stored to LDS;
//   plane z - 2 of the intermediate goes into the rows of D likewise, and plane z - 3 of D is whole and stored.
// A plane thus is in LDS once and read (Q + 2) / Q times a line, three lines a point, where runs that gather whole rows hold three planes and read
// every entry's row: 27 reads a point, and as long a list of them.  A point goes into three rows of the same x and y at once, which is what
// v_mfma_f32_4x4x1 does: four values, broadcast from the block of lanes that the instruction names, times the value of each lane, added to four registers,
// each sum rounded once as by a fused multiply-add (5 million random ones, denormals and infinities among them, have fmaf's bits) -- a row's entries come in
// the order of its columns, so results carry the reference's bits.  The fourth register is left over; three fused multiply-adds in 8.8 cycles are still
// more than v_fmac_f32 with a DPP broadcast makes (4.6 each).  96^3 points, N = 64: 164 us (174 on another card), against 533 in gathering runs and 550 as two products;
// on DPP in this arrangement 216.  What is left, of 174: the matrix cores are busy 0.43 of the time, other VALU work and their power take as much again;
// without any loads it takes 127, without the sums 150.  (A plane of C ahead of time into L2: nothing gained.  Each row's values in three parts, as the
// planes ask for them, 180.  Lines of seven points: registers spill, 424.)
template <int Q, bool ACC, bool WIDE>
__global__ __launch_bounds__(kBoxBlock) void fused_box_kernel(const BoxArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int run = xcd_contiguous(blockIdx.x, a.per_xcd);
  if (run >= a.n_runs) return;
  constexpr int BX = 2 * Q, TW = BX + 2, CW = BX + 4, ROW = 256, WAVES = kBoxBlock / 64;
  const int c0 = run % a.strips * 64, r1 = run / a.strips, r2 = r1 / a.tx;
  const int x0 = r1 % a.tx * BX, y0 = r2 % a.ty * a.by, z0 = r2 / a.ty * a.zlen, z1 = min(a.nz, z0 + a.zlen);
  if (z0 >= z1) return;
  const int nx = a.nx, ny = a.ny, nz = a.nz, N = a.N, by = a.by;
  const int c_lines = by + 4, t_lines = by + 2, c_bytes = CW * ROW * c_lines, t_bytes = TW * ROW * t_lines, t_at = 2 * c_bytes, v_at = t_at + 2 * t_bytes;
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
  // points outside the grid and columns past N are zeros for good
  for (int i = threadIdx.x * 4; i < t_at + 2 * t_bytes; i += kBoxBlock * 4) lds_write(lds0 + i, 0.f);

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, line = wave / 2, half = wave % 2;
  const bool col_ok = c0 + lane < N;
  const int tx = x0 - 1 + half * (Q + 1), ty = y0 - 1 + line, dx = x0 + half * Q, dy = y0 + line;
  const bool t_on = line < t_lines, d_on = line < by;
  BoxValues<Q + 1> tv;
  BoxValues<Q> dv;
  tv.init(a.Bx, a.val_bytes, tx, ty, a, lane, t_on);
  dv.init(a.Ax, a.val_bytes, dx, dy, a, lane, d_on);

  // C's planes: four points (with WIDE) or one to an instruction
  constexpr int POINTS = WIDE ? 4 : 1, kLoads = (CW * (kBoxMaxY + 4) / POINTS + WAVES - 1) / WAVES;
  unsigned from[WIDE ? kLoads : 1];  // bytes from the start of the plane; ~0: nothing there
  auto source = [&](int i) __attribute__((always_inline)) -> unsigned {
    const int s = POINTS * (wave + WAVES * i) + (WIDE ? lane / 16 : 0), c = c0 + (WIDE ? lane % 16 * 4 : lane), x = x0 - 2 + s % CW, y = y0 - 2 + s / CW;
    return s < CW * c_lines && x >= 0 && x < nx && y >= 0 && y < ny && c < N ? 4u * (((unsigned)y * nx + x) * N + c) : ~0u;
  };
  if constexpr (WIDE) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) from[i] = source(i);
  }
  auto fetch = [&](int z) __attribute__((always_inline)) {
    if (z >= nz || z > z1 + 1) return;
    const float *base = a.C + (size_t)z * nx * ny * N;
    const unsigned to = lds0 + (z & 1) * c_bytes + wave * (POINTS * ROW);
    // (written out: for loads into LDS that it knows of the compiler has every later read of LDS wait.  Nobody else counts the states that must pass
    // before the load reads its base, which may come from a lane of a register (five), and m0 (one).)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // (m0 named as overwritten: of a reserved register worth a warning)
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const unsigned f = WIDE ? from[WIDE ? i : 0] : source(i);
      if (f != ~0u) {
        if constexpr (WIDE) asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to + i * (WAVES * POINTS * ROW)), "v"(f), "s"(base) : "memory", "m0");
        else asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dword %1, %2" ::"s"(to + i * (WAVES * POINTS * ROW)), "v"(f), "s"(base) : "memory", "m0");
      }
    }
#pragma clang diagnostic pop
  };

  // acc[q][i]: the sum of point q's row in plane z - 1 + i of the three that read plane z
  acc4 at[Q + 1], ad[Q];
#pragma unroll
  for (int q = 0; q <= Q; ++q) at[q] = 0.f;
#pragma unroll
  for (int q = 0; q < Q; ++q) ad[q] = 0.f;
  // a plane's part in the sums of the rows below it, in it and above it, in the order of the rows' entries
  auto add_plane = [&](auto &acc, unsigned values, unsigned from_lds, auto width) __attribute__((always_inline)) {
    constexpr int W = decltype(width)::value, P = sizeof(acc) / sizeof(acc[0]) + 2;
    float v[P - 2];
#pragma unroll
    for (int q = 0; q < P - 2; ++q) v[q] = lds_read(values + q * 36);
    static_for<0, 3>([&](auto yc) __attribute__((always_inline)) {
      constexpr int jy = decltype(yc)::value;
      float x[P];
#pragma unroll
      for (int p = 0; p < P; ++p) x[p] = lds_read(from_lds + (jy * W + p) * ROW);
      static_for<0, P>([&](auto pc) __attribute__((always_inline)) {
        static_for<0, 3>([&](auto xc) __attribute__((always_inline)) {
          constexpr int p = decltype(pc)::value, jx = 2 - decltype(xc)::value, q = p - jx;
          if constexpr (q >= 0 && q < P - 2) acc[q] = __builtin_amdgcn_mfma_f32_4x4x1f32(v[q], x[p], acc[q], 4, jy * 3 + jx, 0);
        });
      });
    });
  };

  const int zs = max(0, z0 - 2), t_first = max(0, z0 - 1), t_last = min(nz - 1, z1);
  const unsigned c_read = lds0 + ((t_on ? line : 0) * CW + half * (Q + 1)) * ROW + lane * 4;
  const unsigned t_write = lds0 + t_at + ((t_on ? line : 0) * TW + half * (Q + 1)) * ROW + lane * 4;
  const unsigned t_read = lds0 + t_at + ((d_on ? line : 0) * TW + half * Q) * ROW + lane * 4;
  __syncthreads();
  fetch(zs);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    tv.load(zs - 1 + i, lane);
    dv.load(zs - 3 + i, lane);
    tv.turn();
    dv.turn();
  }
  tv.load(zs + 1, lane);
  dv.load(zs - 1, lane);
  const unsigned tv_at = lds0 + v_at + wave * (BoxValues<Q + 1>::kBytes + BoxValues<Q>::kBytes), dv_at = tv_at + BoxValues<Q + 1>::kBytes;
  const unsigned tv_read = BoxValues<Q + 1>::place(tv_at, lane), dv_read = BoxValues<Q>::place(dv_at, lane);
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  tv.put(tv_at, lane);
  dv.put(dv_at, lane);
  __syncthreads();
  for (int z = zs; z <= z1 + 2; ++z) {
    fetch(z + 1);
    tv.load(z + 2, lane);
    dv.load(z, lane);
    if (z < nz && t_on) add_plane(at, tv_read, c_read + (z & 1) * c_bytes, std::integral_constant<int, CW>{});
    if (z - 1 >= t_first && z - 1 <= t_last && t_on && ty >= 0 && ty < ny) {
      const unsigned to = t_write + (~z & 1) * t_bytes;
#pragma unroll
      for (int q = 0; q <= Q; ++q)
        if (tx + q >= 0 && tx + q < nx) lds_write(to + q * ROW, at[q][0]);
    }
    const int zt = z - 2, zd = z - 3;
    if (zt >= t_first && zt <= t_last && d_on) add_plane(ad, dv_read, t_read + (z & 1) * t_bytes, std::integral_constant<int, TW>{});
    // the next plane of C is there, and so are the values, before younger stores
    __builtin_amdgcn_s_waitcnt(0x0f70);
    tv.put(tv_at, lane);
    dv.put(dv_at, lane);
    if (zd >= z0 && zd < z1 && d_on && dy < ny && col_ok) {
      float *out = a.D + (((size_t)zd * ny + dy) * nx + dx) * N + c0 + lane;
#pragma unroll
      for (int q = 0; q < Q; ++q)
        if (dx + q < nx) __builtin_nontemporal_store(ACC ? out[(size_t)q * N] + ad[q][0] : ad[q][0], out + (size_t)q * N);
    }
#pragma unroll
    for (int q = 0; q <= Q; ++q) at[q] = acc4{at[q][1], at[q][2], 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < Q; ++q) ad[q] = acc4{ad[q][1], ad[q][2], 0.f, 0.f};
    lds_barrier();
  }
}

hipError_t launch_fused_box(BoxArgs a, int accumulate, hipStream_t st) {
  const int lds = box_lds(a.q, a.by);
  if (a.by < 1 || a.by > kBoxMaxY || lds > kMaxLds || a.n_runs <= 0) return hipErrorInvalidValue;
  a.per_xcd = per_xcd_of(a.n_runs);
  const dim3 grid(grid_of(a.n_runs));
  const bool wide = a.N % 4 == 0;  // a load of four floats into LDS wants 16 bytes' alignment (operands have it: tf_dense_wrap_device)
  hipError_t err = hipErrorInvalidValue;
#define CALL3(Q_, ACC_, WIDE_)                                                                                                                        \
  do {                                                                                                                                                \
    err = hipFuncSetAttribute(reinterpret_cast<const void *>(fused_box_kernel<Q_, ACC_, WIDE_>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);    \
    if (err == hipSuccess) hipLaunchKernelGGL((fused_box_kernel<Q_, ACC_, WIDE_>), grid, dim3(kBoxBlock), lds, st, a);                                \
  } while (0)
#define CALL(Q_)                                                                            \
  do {                                                                                      \
    if (accumulate) { if (wide) CALL3(Q_, true, true); else CALL3(Q_, true, false); }       \
    else { if (wide) CALL3(Q_, false, true); else CALL3(Q_, false, false); }                \
  } while (0)
  if (a.q == 6) CALL(6);
  else if (a.q == 4) CALL(4);
#undef CALL
#undef CALL3
  return err != hipSuccess ? err : hipGetLastError();
}

}  // namespace tf
