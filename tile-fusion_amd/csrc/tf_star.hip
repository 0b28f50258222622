// Fused SpMM-SpMM on the 7-point stencil of a 3D grid and the 5-point one of a 2D grid (gfx950): D = A (B C), A and B the pattern in which every grid
// point reads itself and its neighbours along the axes, x fastest (checked against the matrices by the inspector: build_box in tf_march.cpp).  Any values.
// The reference's answer to such patterns is tiling with redundancy (fusion/src/SpMM_SpMM.cpp:984-1057).
#include <hip/hip_runtime.h>

#include "tf_internal.h"
#include "tf_device.h"

namespace tf {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
constexpr unsigned kNowhere = 0x80000000u;  // past the end of every buffer: loads give zeros

__device__ __forceinline__ f4 lds_read4(unsigned addr) { return *reinterpret_cast<const __attribute__((address_space(3))) f4 *>(addr); }
__device__ __forceinline__ void lds_write4(unsigned addr, const f4 &v) { *reinterpret_cast<__attribute__((address_space(3))) f4 *>(addr) = v; }

// acc += (lane L of the quad's value) * x
template <int L> __device__ __forceinline__ void fma_quad(float val, const f4 &x, float (&acc)[4]) {
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %4, %5 quad_perm:[%9,%9,%9,%9] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %1, %4, %6 quad_perm:[%9,%9,%9,%9] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %2, %4, %7 quad_perm:[%9,%9,%9,%9] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %3, %4, %8 quad_perm:[%9,%9,%9,%9] row_mask:0xf bank_mask:0xf"
      : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3])
      : "v"(val), "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "n"(L));
}

// A row's values: lane l of a quad holds the ones of the neighbours l and 4 + l of (-z, -y, -x, itself, +x, +y, +z), zero for a neighbour that is not there.
struct StarRow { float lo, hi; };
template <bool FLAT>
__device__ __forceinline__ f4 star_sum(const StarRow &v, const f4 &mz, const f4 &my, const f4 &mx, const f4 &own, const f4 &px, const f4 &py, const f4 &pz) {
  float acc[4] = {0.f, 0.f, 0.f, 0.f};  // in the order of the row's entries
  fma_quad<0>(v.lo, mz, acc);
  if constexpr (!FLAT) fma_quad<1>(v.lo, my, acc);
  fma_quad<2>(v.lo, mx, acc);
  fma_quad<3>(v.lo, own, acc);
  fma_quad<0>(v.hi, px, acc);
  if constexpr (!FLAT) fma_quad<1>(v.hi, py, acc);
  fma_quad<2>(v.hi, pz, acc);
  return f4{acc[0], acc[1], acc[2], acc[3]};
}

// Where the rows of the point (x, y) lie among the matrices' values, which both have in the same places.
struct StarPlace {
  unsigned lo, hi;       // byte offsets of the lane's two values, for plane 1 of many
  unsigned first, last;  // ... and by how much less in plane 0 and in the last one
  __device__ __forceinline__ void init(int x, int y, int nx, int ny, int plane, int l) {
    const bool there = x >= 0 && x < nx && y >= 0 && y < ny;
    // entries of plane 0, and those before the point's row in plane 1 (of many): 7 a row, less the ones that fall off the grid
    const int per_plane = 7 * nx * ny - 2 * nx - 2 * ny;
    const int before = 7 * (y * nx + x) - (y + (x > 0)) - y - (y > 0 ? nx : x) - (y == ny - 1 ? x : 0);
    const int row = per_plane - nx * ny + before;
    const int at_y = 1, at_x = at_y + (y > 0), own = at_x + (x > 0), at_px = own + 1, at_py = at_px + (x < nx - 1), at_pz = at_py + (y < ny - 1);
    const int k_lo = l == 0 ? 0 : l == 1 ? at_y : l == 2 ? at_x : own, k_hi = l == 0 ? at_px : l == 1 ? at_py : at_pz;
    const bool has_lo = l == 0 || l == 3 || (l == 1 ? y > 0 : x > 0), has_hi = l == 2 || (l == 0 ? x < nx - 1 : l == 1 && y < ny - 1);
    lo = there && has_lo ? 4u * (unsigned)(row + k_lo) : kNowhere;
    hi = there && has_hi ? 4u * (unsigned)(row + k_hi) : kNowhere;
    // in plane 0 the rows before this one in the plane have an entry less each, and so has this one in front of any of its others
    first = 4u * (unsigned)(row - (before - (y * nx + x)) + 1);
    last = 4u * (unsigned)(y * nx + x);
  }
  __device__ __forceinline__ StarRow load(__amdgpu_buffer_rsrc_t from, int z, int nz, int per_plane, int l) const {
    unsigned a = lo, b = hi;
    int so = 0;
    if (z >= 1 && z <= nz - 2) {
      so = (z - 1) * 4 * per_plane;
    } else {
      const bool out = z < 0 || z >= nz;
      const unsigned less = z == 0 ? first : last;
      if (z > 0 && !out) so = (nz - 2) * 4 * per_plane;
      a = out || a >= kNowhere || (z == 0 && l == 0) ? kNowhere : a - less;
      b = out || b >= kNowhere || (z > 0 && l == 2) ? kNowhere : b - less;
    }
    return {__uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(from, (int)a, so, 0)), __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(from, (int)b, so, 0))};
  }
};

}  // namespace

// A run is a column of 16 x by grid points and a range of planes, 32 columns of C wide; a workgroup walks it plane by plane.  A lane group of eight holds
// two neighbouring points (x, y), (x + 1, y) of the intermediate -- the column and one point around it -- for the whole run, four columns a lane: what lies
// above and below them is in its own registers, of C as of the intermediate, and what lies beside them comes through LDS.  Step z makes plane z of the
// intermediate of the planes z - 1, z, z + 1 of C, and plane z - 1 of D likewise, while plane z + 1 of C goes to LDS and planes z + 2 and
// z + 3 are on their way to registers; one barrier a step.  The points around those of the intermediate pass through a register to LDS.
// No lists: a row's place among the values follows from its point; where A and B are one matrix a row's values are kept from the step that makes the
// intermediate to the one that makes D (128^3 points, N = 64: 221 us, 250 with a load for each).  Bound: HBM, 1.26 GB at 5.7 TB/s, more than a plain copy's 5.0
// (gathering runs over lists 290, two products 604; the clocks that launches in close order leave make it 260); on 64^3 points, N = 64, 33 us (49, 56), the steps
// themselves, 1.4 us each.
// 16 by 8 points of 32 columns: the intermediate 1.4 times and C's planes 1.8 times the column, where 8 by 8 of 64 columns are 1.5 and 2.1, in
// as much of LDS.  Each sum is made in the order of the row's entries, so results carry
// the reference's bits; what is outside the grid is zero, with zeros for values.
// FLAT: a 2D grid, its lines for planes; a column is up to 94 points of a line, and two workgroups share a compute unit.  (1000 x 1000 points, us, here / as
// two products: N = 64 118 / 292, 100 259 / 522, 128 222 / 556; 900 x 900, N = 32 45 / 82.)
// LDS rows of 128 bytes: two lane groups of a read, two points apart, would meet in the same banks; rows 2 and 3 of every four change places.
template <bool ACC, bool SAME, bool FLAT>
__global__ __launch_bounds__(FLAT ? kFlatBlock : kStarBlock, 3) void fused_star_kernel(const BoxArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int run = xcd_contiguous(blockIdx.x, a.per_xcd);
  if (run >= a.n_runs) return;
  constexpr int LINE = FLAT ? kFlatX + 6 : kStarX + 4, PAIRS = FLAT ? (kFlatX + 2) / 2 : (kStarX + 2) / 2, UP = FLAT ? 0 : LINE * 128;  // UP: bytes from a line to the next
  const int c0 = run % a.strips * 32, r1 = run / a.strips, r2 = r1 / a.tx;
  const int bx = FLAT ? a.bx : kStarX, x0 = r1 % a.tx * bx, y0 = r2 % a.ty * a.by, z0 = r2 / a.ty * a.zlen, z1 = min(a.nz, z0 + a.zlen);
  if (z0 >= z1) return;
  const int nx = a.nx, ny = a.ny, nz = a.nz, N = a.N, by = a.by, plane = nx * ny, per_plane = 7 * plane - 2 * nx - 2 * ny;
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
  const unsigned c_bytes = FLAT ? kFlatLine : kStarLine * (by + 4), t_bytes = FLAT ? kFlatLine : kStarLine * (by + 2);
  const unsigned t_at = 2 * c_bytes - UP;  // (of the intermediate lines 1 .. by + 2 only)
  const int group = threadIdx.x / 8, gl = threadIdx.x % 8, l = gl % 4, col = c0 + gl * 4;
  const int line = FLAT ? 0 : group / PAIRS, pair = FLAT ? group : group % PAIRS, x = x0 - 1 + 2 * pair, y = FLAT ? 0 : y0 - 1 + line;
  const bool t_on = FLAT ? 2 * pair < bx + 2 : line < by + 2, col_ok = col < N;
  auto row_at = [&](int i) __attribute__((always_inline)) { return lds0 + (unsigned)((i ^ (i >> 1 & 1)) * 128 + gl * 16); };
  const int i0 = (FLAT ? 0 : t_on ? line + 1 : 1) * LINE + 1 + 2 * pair;
  const unsigned at_mx = row_at(i0 - 1), at_0 = row_at(i0), at_1 = row_at(i0 + 1), at_px = row_at(i0 + 2);

  // the group's point around those of the intermediate: the lines before and behind, then the ends of the others
  const int around = FLAT ? 2 : 2 * (LINE - 2) + 2 * (by + 2), e = group - 2 * (LINE - 2);
  const int ri = FLAT ? (group == 0 ? 0 : bx + 3) : e < -(LINE - 2) ? group + 1 : e < 0 ? (by + 3) * LINE + 1 + group - (LINE - 2) : (1 + e / 2) * LINE + (e & 1) * (LINE - 1);
  const bool r_on = group < around;
  const unsigned at_r = row_at(ri);

  auto source = [&](int px, int py, bool on) __attribute__((always_inline)) -> unsigned {
    return on && col_ok && px >= 0 && px < nx && py >= 0 && py < ny ? 4u * (((unsigned)py * nx + px) * N + col) : kNowhere;
  };
  const unsigned from0 = source(x, y, t_on), from1 = source(x + 1, y, t_on), from_r = source(x0 - 2 + ri % LINE, FLAT ? 0 : y0 - 2 + ri / LINE, r_on);
  const bool in_0 = t_on && x >= 0 && x < nx && y >= 0 && y < ny, in_1 = t_on && x + 1 >= 0 && x + 1 < nx && y >= 0 && y < ny;
  const bool d_line = (FLAT || (line >= 1 && line <= by)) && y < ny && col_ok;
  const bool d_0 = d_line && pair > 0 && x < min(nx, x0 + bx), d_1 = d_line && x + 1 < min(nx, x0 + bx);
  const int plane_bytes = (int)((unsigned)plane * N * 4u);
  auto c_plane = [&](int z) __attribute__((always_inline)) {  // (a buffer of nothing outside the grid and the run)
    const bool there = z >= 0 && z < nz && z <= z1 + 1;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.C + (there ? (size_t)z * plane * N : 0)), 0, there ? plane_bytes : 0, 0x00020000);
  };
  auto load = [&](__amdgpu_buffer_rsrc_t from, unsigned at) __attribute__((always_inline)) {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    const u4 v = __builtin_amdgcn_raw_buffer_load_b128(from, (int)at, 0, 0);
    return f4{__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3])};
  };
  // (written out: the compiler makes one store of the two branches and drops the hint; the state that must pass before its registers are written is then ours too)
  auto store = [&](f4 *to, const f4 &v) __attribute__((always_inline)) {
    if (a.streaming) asm volatile("global_store_dwordx4 %0, %1, off nt\n\ts_nop 0" ::"v"(to), "v"(v) : "memory");
    else *to = v;
  };
  const __amdgpu_buffer_rsrc_t av = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.Ax), 0, (int)a.val_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t bv = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.Bx), 0, (int)a.val_bytes, 0x00020000);
  StarPlace p0, p1;
  p0.init(t_on ? x : -1, y, nx, ny, plane, l);
  p1.init(t_on ? x + 1 : -1, y, nx, ny, plane, l);

  // planes of C: slot (z - zs + 1) mod 4; around them: slot (z - zs - 1) mod 2; values: mod 2
  const int zs = max(0, z0 - 1), t_last = min(nz - 1, z1);
  f4 c[4][2], r[2], t1[2] = {0.f, 0.f}, t2[2] = {0.f, 0.f};  // t1, t2: the intermediate one and two planes back
  StarRow vb[2][2], va[2][2];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const auto from = c_plane(zs - 1 + i);
    c[i][0] = load(from, from0);
    c[i][1] = load(from, from1);
    if (i == 1) r[1] = load(from, from_r);
  }
  if (t_on) {
    lds_write4(at_0, c[1][0]);
    lds_write4(at_1, c[1][1]);
  }
  if (r_on) lds_write4(at_r, r[1]);
  r[0] = load(c_plane(zs + 1), from_r);
  r[1] = load(c_plane(zs + 2), from_r);
  vb[0][0] = p0.load(bv, zs, nz, per_plane, l);
  vb[0][1] = p1.load(bv, zs, nz, per_plane, l);
  va[0][0] = p0.load(av, zs - 1, nz, per_plane, l);
  va[0][1] = p1.load(av, zs - 1, nz, per_plane, l);
  lds_barrier();

  auto step = [&](int z, auto phase) __attribute__((always_inline)) {
    constexpr int P = decltype(phase)::value, M = P % 4, O = (P + 1) % 4, U = (P + 2) % 4, B = P % 2;  // slots of planes z - 1, z, z + 1
    const unsigned c_now = B * c_bytes, c_next = (1 - B) * c_bytes, t_now = t_at + B * t_bytes, t_back = t_at + (1 - B) * t_bytes;
    vb[1 - B][0] = p0.load(bv, z + 1, nz, per_plane, l);
    vb[1 - B][1] = p1.load(bv, z + 1, nz, per_plane, l);
    if constexpr (!SAME) {
      va[1 - B][0] = p0.load(av, z, nz, per_plane, l);
      va[1 - B][1] = p1.load(av, z, nz, per_plane, l);
    }
    f4 t[2] = {0.f, 0.f};
    if (z <= t_last) {
      const f4 s0 = star_sum<FLAT>(vb[B][0], c[M][0], lds_read4(at_0 + c_now - UP), lds_read4(at_mx + c_now), c[O][0], c[O][1], lds_read4(at_0 + c_now + UP), c[U][0]);
      const f4 s1 = star_sum<FLAT>(vb[B][1], c[M][1], lds_read4(at_1 + c_now - UP), c[O][0], c[O][1], lds_read4(at_px + c_now), lds_read4(at_1 + c_now + UP), c[U][1]);
      t[0] = in_0 ? s0 : f4(0.f);
      t[1] = in_1 ? s1 : f4(0.f);
    }
    {  // the slot of plane z - 1 takes plane z + 3
      const auto from = c_plane(z + 3);
      c[M][0] = load(from, from0);
      c[M][1] = load(from, from1);
    }
    if (t_on) {
      lds_write4(at_0 + t_now, t[0]);
      lds_write4(at_1 + t_now, t[1]);
      lds_write4(at_0 + c_next, c[U][0]);
      lds_write4(at_1 + c_next, c[U][1]);
    }
    if (r_on) lds_write4(at_r + c_next, r[B]);
    r[B] = load(c_plane(z + 3), from_r);
    if (z - 1 >= z0 && t_on) {
      const f4 d0 = star_sum<FLAT>(va[B][0], t2[0], lds_read4(at_0 + t_back - UP), lds_read4(at_mx + t_back), t1[0], t1[1], lds_read4(at_0 + t_back + UP), t[0]);
      const f4 d1 = star_sum<FLAT>(va[B][1], t2[1], lds_read4(at_1 + t_back - UP), t1[0], t1[1], lds_read4(at_px + t_back), lds_read4(at_1 + t_back + UP), t[1]);
      f4 *out = reinterpret_cast<f4 *>(a.D + (((size_t)(z - 1) * ny + y) * nx + x) * N + col);
      f4 *out1 = reinterpret_cast<f4 *>(a.D + (((size_t)(z - 1) * ny + y) * nx + x + 1) * N + col);
      if (d_0) store(out, ACC ? *out + d0 : d0);
      if (d_1) store(out1, ACC ? *out1 + d1 : d1);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      t2[q] = t1[q];
      t1[q] = t[q];
      if constexpr (SAME) va[1 - B][q] = vb[B][q];
    }
    lds_barrier();
  };
  for (int z = zs; z <= z1; z += 4) {
    step(z, std::integral_constant<int, 0>{});
    if (z + 1 > z1) break;
    step(z + 1, std::integral_constant<int, 1>{});
    if (z + 2 > z1) break;
    step(z + 2, std::integral_constant<int, 2>{});
    if (z + 3 > z1) break;
    step(z + 3, std::integral_constant<int, 3>{});
  }
}

hipError_t launch_fused_star(BoxArgs a, int accumulate, hipStream_t st) {
  const bool flat = a.ny == 1;
  const int lds = flat ? flat_lds() : star_lds(a.by), block = flat ? kFlatBlock : kStarBlock;
  if (a.by < 1 || a.by > kStarMaxY || a.bx < 1 || a.bx > (flat ? kFlatX : kStarX) || a.N % 4 != 0 || a.n_runs <= 0) return hipErrorInvalidValue;
  a.per_xcd = per_xcd_of(a.n_runs);
  // Streaming stores but where strips share lines of a D that the Infinity Cache does not hold, which would go to memory in parts (us, streaming / plain:
  // N = 100, 128^3 points 718 / 642, 1000 x 1000 302 / 259, 64^3 55.5 / 56.7; N = 84, 96^3 201 / 204; N = 48, 64^3 32.0 / 33.3; whole lines, N = 64, 128^3 220 / 229, 96^3
  // 107 / 121, 1000 x 1000 118 / 120.  On the wrong side by 3 and 4 %: 128^3, N = 48 241 / 249, N = 32 122 / 117).
  a.streaming = a.N % 32 == 0 || (long long)a.nx * a.ny * a.nz * a.N * 4 <= (320ll << 20);
  const dim3 grid(grid_of(a.n_runs));
#define CALL(ACC_, SAME_, FLAT_)                                                                                                                             \
  do {                                                                                                                                                      \
    const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void *>(fused_star_kernel<ACC_, SAME_, FLAT_>), hipFuncAttributeMaxDynamicSharedMemorySize, lds); \
    if (err != hipSuccess) return err;                                                                                                                      \
    hipLaunchKernelGGL((fused_star_kernel<ACC_, SAME_, FLAT_>), grid, dim3(block), lds, st, a);                                                              \
  } while (0)
#define CALL2(ACC_, SAME_) do { if (flat) CALL(ACC_, SAME_, true); else CALL(ACC_, SAME_, false); } while (0)
  if (a.Ax == a.Bx) { if (accumulate) CALL2(true, true); else CALL2(false, true); }
  else { if (accumulate) CALL2(true, false); else CALL2(false, false); }
#undef CALL2
#undef CALL
  return hipGetLastError();
}

}  // namespace tf
