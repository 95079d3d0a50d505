// otm_coarse_dev.hpp -- device bodies of the coarse multigrid levels
// (stored 27-point stencils, transfers, coarsest solve), shared by the
// single-cell launches (otm_coarse.hip) and the batched multi-cell launches
// (otm_batch.hip).
//
// Stencil layout: st[o*nn + v] couples node v to v + off(o) with
// off(o) = (o%3-1, o/3%3-1, o/9-1); o = 13 is the diagonal (the reference
// keeps 27 SoA arrays the same way, grid.cpp:189-220, diagonal at index 13,
// grid.cu:707-809).
//
// Galerkin coarse operators A_{l+1} = P^T A_l P with trilinear P
// (grid.cu:811-940, grid_ex.cu:16-227) are formed element by element: a
// coarse element's 8x8 matrix is the sum over its 8 children c of
// Q_c^T E_c Q_c, where Q_c interpolates the coarse element's corners to the
// child's corners. This equals the stencil-level triple product exactly.
#pragma once
#include "otm_kernels.hpp"

namespace otm {

__device__ inline long long lin(const Geom& g, int x, int y, int z) {
  return (long long)x + (long long)g.nx * ((long long)y + (long long)g.ny * z);
}

// ---- per-node operations of the stored-stencil levels ----
// Stencil entries of node v. FP16 storage (HALF) keeps the 26 couplings
// divided by a per-level scale; the diagonal is rebuilt as minus their sum,
// so rows keep a zero sum and the constants stay in the null space.
template <bool HALF>
__device__ inline void load_stencil(const StRef& S, long long nn, long long v, float a[27]) {
  if constexpr (HALF) {
    const float sc = *S.scale;
    float off = 0.f;
#pragma unroll
    for (int o = 0; o < 27; o++) {
      if (o == 13) continue;
      a[o] = (float)S.f16[o * nn + v] * sc;
      off += a[o];
    }
    a[13] = -off;
  } else {
#pragma unroll
    for (int o = 0; o < 27; o++) a[o] = S.f32[o * nn + v];
  }
}

// GS update at node (x,y,z): u = (f - sum_{o != 13} a_o u_o) / a_13.
template <bool HALF>
__device__ inline void st_gs_node(const Geom& g, const StRef& S, const float* __restrict__ f, float* u, int x, int y,
                                  int z) {
  const long long v = lin(g, x, y, z);
  const int xs[3] = {x == 0 ? g.nx - 1 : x - 1, x, x == g.nx - 1 ? 0 : x + 1};
  const int ys[3] = {y == 0 ? g.ny - 1 : y - 1, y, y == g.ny - 1 ? 0 : y + 1};
  const int zs[3] = {z == 0 ? g.nz - 1 : z - 1, z, z == g.nz - 1 ? 0 : z + 1};
  float a[27];
  load_stencil<HALF>(S, g.nn, v, a);
  const float inv = 1.f / a[13];
#pragma unroll
  for (int k = 0; k < OTM_NRHS; k++) {
    const float* uk = u + k * g.nn;
    float s = 0.f;
#pragma unroll
    for (int o = 0; o < 27; o++) {
      if (o == 13) continue;
      s += a[o] * uk[lin(g, xs[o % 3], ys[(o / 3) % 3], zs[o / 9])];
    }
    u[k * g.nn + v] = (f[k * g.nn + v] - s) * inv;
  }
}

// res = f - A u at node t.
template <bool HALF>
__device__ inline void st_resid_node(const Geom& g, const StRef& S, const float* __restrict__ f, const float* u,
                                     float* res, long long t) {
  int x, y, z;
  split_node(g.nx, g.ny, t, x, y, z);
  const int xs[3] = {x == 0 ? g.nx - 1 : x - 1, x, x == g.nx - 1 ? 0 : x + 1};
  const int ys[3] = {y == 0 ? g.ny - 1 : y - 1, y, y == g.ny - 1 ? 0 : y + 1};
  const int zs[3] = {z == 0 ? g.nz - 1 : z - 1, z, z == g.nz - 1 ? 0 : z + 1};
  float a[27];
  if constexpr (HALF) {
    load_stencil<HALF>(S, g.nn, t, a);
  } else {
#pragma unroll
    for (int o = 0; o < 27; o++) a[o] = ld_off(S.f32 + (size_t)o * (size_t)g.nn, 4u * (unsigned)t);
  }
  // neighbour byte offsets from wave-uniform bases in 32 bits (64-bit
  // per-neighbour addresses were half of this kernel's instructions)
  const unsigned nx = (unsigned)g.nx, nxy = (unsigned)g.nx * (unsigned)g.ny;
  unsigned off[27];
#pragma unroll
  for (int o = 0; o < 27; o++)
    off[o] = 4u * ((unsigned)xs[o % 3] + nx * (unsigned)ys[(o / 3) % 3] + nxy * (unsigned)zs[o / 9]);
#pragma unroll
  for (int k = 0; k < OTM_NRHS; k++) {
    const float* uk = u + (size_t)k * (size_t)g.nn;
    float s = 0.f;
#pragma unroll
    for (int o = 0; o < 27; o++) s += a[o] * ld_off(uk, off[o]);
    res[k * g.nn + t] = f[k * g.nn + t] - s;
  }
}

// f_c(I) = sum_{d in {-1,0,1}^3} w(d) res(2I + d), w = prod(d_i == 0 ? 1 : 1/2)
// (restrict_residual_kernel_H, grid.cu:811-878, weights (2-|d|)/2 per axis).
__device__ inline void restrict_node(const Geom& fg, const Geom& cg, const float* res, float* fc, long long t) {
  int X, Y, Z;
  split_node(cg.nx, cg.ny, t, X, Y, Z);
  const int x = 2 * X, y = 2 * Y, z = 2 * Z;
  const int xs[3] = {x == 0 ? fg.nx - 1 : x - 1, x, x + 1};
  const int ys[3] = {y == 0 ? fg.ny - 1 : y - 1, y, y + 1};
  const int zs[3] = {z == 0 ? fg.nz - 1 : z - 1, z, z + 1};
  const float w1[3] = {0.5f, 1.f, 0.5f};
  // byte offsets in 32 bits from wave-uniform bases
  unsigned rb[9];
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int b = 0; b < 3; b++) rb[b + 3 * c] = (unsigned)fg.nx * ((unsigned)ys[b] + (unsigned)fg.ny * (unsigned)zs[c]);
#pragma unroll
  for (int k = 0; k < OTM_NRHS; k++) {
    const float* rk = res + (size_t)k * (size_t)fg.nn;
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int b = 0; b < 3; b++) {
        float row = 0.f;
#pragma unroll
        for (int a = 0; a < 3; a++) row += w1[a] * ld_off(rk, 4u * (rb[b + 3 * c] + (unsigned)xs[a]));
        s += w1[b] * w1[c] * row;
      }
    fc[k * cg.nn + t] = s;
  }
}

// Restriction with 8 lanes per coarse node for small coarse levels (the
// same weights; lane j takes the fine offsets o = j + 8q, the group adds
// with group8_sum, lanes 0-2 write). Thread t serves coarse node t / 8.
constexpr long long kRestrict8MaxNodes = 4096;
__host__ __device__ inline bool restrict8(const Geom& cg) { return cg.nn <= kRestrict8MaxNodes; }
__device__ inline void restrict8_body(const Geom& fg, const Geom& cg, const float* __restrict__ res,
                                      float* __restrict__ fc, long long t) {
  const long long node = t >> 3;
  const int j = (int)(t & 7);
  if (node >= cg.nn) return;
  int X, Y, Z;
  split_node(cg.nx, cg.ny, node, X, Y, Z);
  const int x = 2 * X, y = 2 * Y, z = 2 * Z;
  float a[OTM_NRHS] = {0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int o = j + 8 * q;
    if (o < 27) {
      const int dx = o % 3 - 1, dy = (o / 3) % 3 - 1, dz = o / 9 - 1;
      const float w = (dx ? 0.5f : 1.f) * (dy ? 0.5f : 1.f) * (dz ? 0.5f : 1.f);
      const unsigned off = 4u * ((unsigned)wrapm(x + dx, fg.nx) +
                                 (unsigned)fg.nx * ((unsigned)wrapm(y + dy, fg.ny) + (unsigned)fg.ny * (unsigned)wrapm(z + dz, fg.nz)));
#pragma unroll
      for (int k = 0; k < OTM_NRHS; k++) a[k] += w * ld_off(res + (size_t)k * (size_t)fg.nn, off);
    }
  }
#pragma unroll
  for (int k = 0; k < OTM_NRHS; k++) a[k] = group8_sum(a[k]);
  if (j < OTM_NRHS) fc[(size_t)j * (size_t)cg.nn + node] = j == 0 ? a[0] : (j == 1 ? a[1] : a[2]);
}

// ---- per-level bodies ----
// GS update of one of 8 colours (parity of x, y, z), colour = cx + 2cy + 4cz.
template <bool HALF>
__device__ inline void st_gs_color_body(const Geom& g, const StRef& S, const float* __restrict__ f, float* u, int cx,
                                        int cy, int cz, long long t) {
  const int hx = g.nx >> 1, hy = g.ny >> 1, hz = g.nz >> 1;
  const long long cnt = (long long)hx * hy * hz;
  if (t >= cnt) return;
  int x, y, z;
  split_node(hx, hy, t, x, y, z);
  x = 2 * x + cx;
  y = 2 * y + cy;
  z = 2 * z + cz;
  st_gs_node<HALF>(g, S, f, u, x, y, z);
}

// Levels up to this many nodes take the 8-lanes-per-node residual (latency
// bound: 10 -> 3.4-5.4 us at 16^3 and 32^3); larger ones one node per thread
// (at 64^3 the 8-lane form's stencil reads coalesce worse: 12.7 -> 26 us).
constexpr long long kResid8MaxNodes = 65536;
__host__ __device__ inline bool st_resid8(const Geom& g, bool half) { return !half && g.nn <= kResid8MaxNodes; }

// res = f - A u with 8 lanes per node (FP32 stencils): lane j of a group
// takes the entries o = j, j + 8, j + 16, j + 24 (o < 27) with their three
// load cases' neighbours, the group adds its partial sums (group8_sum) and
// lanes 0-2 write. Thread t serves node t / 8 (a whole group is past the
// level when its node is). One node per thread left small levels waiting
// on its 111 loads one after another (10 us at 16^3 and 32^3).
__device__ inline void st_residual8_body(const Geom& g, const float* __restrict__ st, const float* __restrict__ f,
                                         const float* __restrict__ u, float* __restrict__ res, long long t) {
  const long long node = t >> 3;
  const int j = (int)(t & 7);
  if (node >= g.nn) return;
  int x, y, z;
  split_node(g.nx, g.ny, node, x, y, z);
  const unsigned nx = (unsigned)g.nx, nxy = (unsigned)g.nx * (unsigned)g.ny;
  float a[OTM_NRHS] = {0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int o = j + 8 * q;
    if (o < 27) {
      const float c = ld_off(st + (size_t)o * (size_t)g.nn, 4u * (unsigned)node);
      const unsigned w = 4u * ((unsigned)wrapm(x + o % 3 - 1, g.nx) + nx * (unsigned)wrapm(y + (o / 3) % 3 - 1, g.ny) +
                               nxy * (unsigned)wrapm(z + o / 9 - 1, g.nz));
#pragma unroll
      for (int k = 0; k < OTM_NRHS; k++) a[k] += c * ld_off(u + (size_t)k * (size_t)g.nn, w);
    }
  }
#pragma unroll
  for (int k = 0; k < OTM_NRHS; k++) a[k] = group8_sum(a[k]);
  if (j < OTM_NRHS) {
    const float s = j == 0 ? a[0] : (j == 1 ? a[1] : a[2]);
    res[(size_t)j * (size_t)g.nn + node] = f[(size_t)j * (size_t)g.nn + node] - s;
  }
}

template <bool HALF>
__device__ inline void st_residual_body(const Geom& g, const StRef& S, const float* __restrict__ f,
                                        const float* __restrict__ u, float* __restrict__ res, long long t) {
  if (t >= g.nn) return;
  st_resid_node<HALF>(g, S, f, u, res, t);
}

// restrict_node when coarse rows are whole waves (cg.nx a multiple of 64,
// t = this wave's first coarse node + lane): a lane loads the fine pair
// (2X, 2X+1) of each of its nine rows as one 8-byte load (a wave reads 512
// contiguous bytes) and takes 2X-1 from the lane before it by DPP; lane 0
// loads it. The same terms in the same order: the same bits.
__device__ inline void restrict_node_pairs(const Geom& fg, const Geom& cg, const float* res, float* fc, long long t) {
  int X, Y, Z;
  split_node(cg.nx, cg.ny, t, X, Y, Z);
  const int x = 2 * X, y = 2 * Y, z = 2 * Z;
  const int xm = x == 0 ? fg.nx - 1 : x - 1;
  const int ys[3] = {y == 0 ? fg.ny - 1 : y - 1, y, y + 1};
  const int zs[3] = {z == 0 ? fg.nz - 1 : z - 1, z, z + 1};
  const float w1[3] = {0.5f, 1.f, 0.5f};
  const bool lane0 = (threadIdx.x & 63) == 0;
  unsigned rb[9];
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int b = 0; b < 3; b++) rb[b + 3 * c] = (unsigned)fg.nx * ((unsigned)ys[b] + (unsigned)fg.ny * (unsigned)zs[c]);
#pragma unroll
  for (int k = 0; k < OTM_NRHS; k++) {
    const float* rk = res + (size_t)k * (size_t)fg.nn;
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int b = 0; b < 3; b++) {
        const unsigned r = rb[b + 3 * c];
        const float2 v = *(const float2*)((const char*)rk + 4u * (r + (unsigned)x));
        float left = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v.y), 0x138, 0xF, 0xF, false));
        if (lane0) left = ld_off(rk, 4u * (r + (unsigned)xm));
        float row = 0.f;
        row += w1[0] * left;
        row += w1[1] * v.x;
        row += w1[2] * v.y;
        s += w1[b] * w1[c] * row;
      }
    fc[k * cg.nn + t] = s;
  }
}

// One thread per coarse node (t); the grid covers whole waves, so the
// paired form may be taken whenever coarse rows are whole waves.
__device__ inline void restrict_body(const Geom& fg, const Geom& cg, const float* __restrict__ res,
                                     float* __restrict__ fc, long long t) {
  if (cg.nx % 64 == 0 && blockDim.x % 64 == 0) {
    if (t < cg.nn) restrict_node_pairs(fg, cg, res, fc, t);
    return;
  }
  if (t >= cg.nn) return;
  restrict_node(fg, cg, res, fc, t);
}

// u_f(i) += sum_I P(i, I) u_c(I), trilinear (prolongate_correction_kernel_H,
// grid.cu:881-940), by coarse cell: thread t owns coarse node (X, Y, Z) and
// the eight fine nodes (2X+dx, 2Y+dy, 2Z+dz). It loads the eight coarse
// values around the cell once per right-hand side and adds to every fine
// node its terms (zero weights skipped): an eighth of the coarse loads of a
// thread per fine node, and paired, coalesced fine accesses. The fine level
// is twice the coarse one along every axis.
__device__ inline void prolong_body(const Geom& fg, const Geom& cg, const float* __restrict__ uc,
                                    float* __restrict__ uf, long long t) {
  if (t >= cg.nn) return;
  int X, Y, Z;
  split_node(cg.nx, cg.ny, t, X, Y, Z);
  const int Xs[2] = {X, X + 1 == cg.nx ? 0 : X + 1};
  const int Ys[2] = {Y, Y + 1 == cg.ny ? 0 : Y + 1};
  const int Zs[2] = {Z, Z + 1 == cg.nz ? 0 : Z + 1};
#pragma unroll
  for (int k = 0; k < OTM_NRHS; k++) {
    const float* ck = uc + k * cg.nn;
    float v[2][2][2];
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int b = 0; b < 2; b++)
#pragma unroll
        for (int a = 0; a < 2; a++)
          v[c][b][a] = ck[(long long)Xs[a] + (long long)cg.nx * ((long long)Ys[b] + (long long)cg.ny * Zs[c])];
    float* fk = uf + k * fg.nn;
#pragma unroll
    for (int dz = 0; dz < 2; dz++)
#pragma unroll
      for (int dy = 0; dy < 2; dy++)
#pragma unroll
        for (int dx = 0; dx < 2; dx++) {
          const ProlongW P = prolong_weights(cg, 2 * X + dx, 2 * Y + dy, 2 * Z + dz);
          float s = 0.f;
#pragma unroll
          for (int c = 0; c < 2; c++)
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
              for (int a = 0; a < 2; a++) {
                const float w = P.wx[a] * P.wy[b] * P.wz[c];
                if (w != 0.f) s += w * v[c & dz][b & dy][a & dx];
              }
          const long long fi = (long long)(2 * X + dx) +
                               (long long)fg.nx * ((long long)(2 * Y + dy) + (long long)fg.ny * (2 * Z + dz));
          fk[fi] += s;
        }
  }
}

// u = Binv f on the coarsest level for the three load cases, FP64
// accumulation: one wave takes two rows of Binv (lanes stride the columns,
// so a row is read in whole cache lines and the load cases' values serve
// both rows) and adds its lanes' sums in a fixed order.
// Bound by reading Binv once, 8 n^2 bytes, and below a few hundred nodes by
// latency. One workgroup inside the tail kernel, a thread per (row, load
// case) walking its row alone, took 6367 us at n = 1331, 479 us at 576 and
// 56 us at 216; spread over the chip 7.5, 4 and 3.5 us.
constexpr int kCoarsestRows = 2 * kWaves;  // rows of one block
__host__ __device__ inline long long coarsest_row_blocks(const Geom& g) {
  return (g.nn + kCoarsestRows - 1) / kCoarsestRows;
}
__device__ inline void coarsest_rows_body(const Geom& g, const double* __restrict__ Binv,
                                          const float* __restrict__ f, float* __restrict__ u, int lb) {
  const int n = (int)g.nn, lane = threadIdx.x & 63;
  const int i0 = lb * kCoarsestRows + 2 * ((int)threadIdx.x >> 6);
  if (i0 >= n) return;
  const int i1 = i0 + 1 < n ? i0 + 1 : i0;
  const double* __restrict__ r0 = Binv + (long long)i0 * n;
  const double* __restrict__ r1 = Binv + (long long)i1 * n;
  double s0[OTM_NRHS] = {0, 0, 0}, s1[OTM_NRHS] = {0, 0, 0};
#pragma unroll 4
  for (int j = lane; j < n; j += 64) {
    const double b0 = r0[j], b1 = r1[j];
#pragma unroll
    for (int k = 0; k < OTM_NRHS; k++) {
      const double fv = (double)f[k * n + j];
      s0[k] += b0 * fv;
      s1[k] += b1 * fv;
    }
  }
#pragma unroll
  for (int k = 0; k < OTM_NRHS; k++) {
    const double v0 = wave_sum(s0[k]), v1 = wave_sum(s1[k]);
    if (lane == 0) {
      u[k * n + i0] = (float)v0;
      u[k * n + i1] = (float)(i1 == i0 ? v0 : v1);
    }
  }
}

// Brick smoother for stored-stencil levels. One workgroup owns an 8^3 brick
// (cut at the level's edge when an edge is not a multiple of 8): u of the
// brick plus a one-node halo sits in LDS. All colours of `sweeps`
// Gauss-Seidel sweeps run inside the brick with workgroup barriers; halo
// values stay frozen at their values on entry (block Gauss-Seidel across
// bricks, exact multicolour Gauss-Seidel inside; a level smaller than a
// brick is smoothed exactly except across its periodic seam). The result
// goes to a second buffer so bricks never read a neighbour's new values. The
// post-smoother runs the colours in reverse order, which is the adjoint of
// the pre-smoother: the V-cycle stays symmetric.
//
// Work split: wave w owns the rows of one (y, z) parity, w = (y%2) + 2(z%2),
// and each of its 64 lanes the node pair (2m, 2m + 1) of one such row, whose
// 2 x 26 couplings it holds in registers (FP16 couplings as loaded, widened
// inside the multiply-adds). The pair's two colours are consecutive in the
// colour order, so one wave does both in a step with no barrier between: the
// eight other rows' values (two 8-byte LDS reads per row and load case) serve
// both nodes, the partner's new value is in a register and the neighbouring
// pair's comes by DPP. A sweep is four steps with one barrier each.
// With a node spread over 8 lanes (each 2 to 4 couplings, partial sums
// added by DPP, 8 steps a sweep) the kernel issued three times the
// instructions and was bound by them: two sweeps at 128^3 (FP16) 97 us, now
// 59; 64^3 (FP16 / FP32) 17 / 13.6, now 14.8 / 13.1.
// Small levels are bound by the latency of the eight steps. There each
// workgroup takes one load case (NR = 1; the couplings are then read three
// times, from L2): a step waits for a third of the reads and multiply-adds.
// 16^3 and 32^3 took 9.2 us with 8 lanes per node. The three load cases
// together (NR = 3) against one per workgroup, FP32 and FP16 stencils, us:
//   bricks   8      64     128    216    256    343    512
//   FP32  8.5 5.6  8.7 6.4  9.1 8.2 10.0 11.4 10.3 12.8 13.6 14.7 13.5 19.1
//   FP16 10.0 5.5 10.3 6.2 10.6 8.2 10.9 10.4 11.4 11.5 13.8 14.1 14.6 21.0
// The line lies where FP16's cross; FP32's cross between 128 and 216 bricks.
// The results have the same bits either way.
constexpr int kBrick = 8;
constexpr int kStBrickThreads = 256;
constexpr int kHalo = kBrick + 2;
// LDS pitches of a row and a plane: the 8-byte reads of half a wave (rows
// two apart, planes two apart) then fall on different banks
constexpr int kStPitch = 12, kStPlane = 144;
constexpr int kStOneMax = 256;  // bricks of a launch up to which NR = 1
__host__ __device__ inline int brick_count(const Geom& g) {
  return ((g.nx + kBrick - 1) / kBrick) * ((g.ny + kBrick - 1) / kBrick) * ((g.nz + kBrick - 1) / kBrick);
}
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// LDS of the brick smoother, one allocation for both stencil precisions
// (a batched launch instantiates both bodies in one kernel).
struct alignas(16) StBrickLds {
  float su[OTM_NRHS][kHalo * kStPlane];  // u of the brick and its halo
};
__device__ inline StBrickLds& st_brick_lds() {
  __shared__ StBrickLds lds;
  return lds;
}

// The brick of block b, its size, and this lane's node pair.
struct StPair {
  int ox, oy, oz, wx, wy, wz;  // first node, edges
  int lx, ly, lz;              // the pair's first node in the brick
  bool act;                    // inside the brick
  unsigned v;                  // its index (of a node of the brick when not)
};
__device__ __forceinline__ StPair st_pair(const Geom& g, int b) {
  StPair P;
  const int bx = (g.nx + kBrick - 1) / kBrick, by = (g.ny + kBrick - 1) / kBrick;
  P.ox = (b % bx) * kBrick;
  P.oy = ((b / bx) % by) * kBrick;
  P.oz = (b / (bx * by)) * kBrick;
  P.wx = min(kBrick, g.nx - P.ox);
  P.wy = min(kBrick, g.ny - P.oy);
  P.wz = min(kBrick, g.nz - P.oz);
  const int m = (int)threadIdx.x & 63, w = (int)threadIdx.x >> 6;
  P.lx = 2 * (m & 3);
  P.ly = 2 * ((m >> 2) & 3) + (w & 1);
  P.lz = 2 * (m >> 4) + (w >> 1);
  P.act = P.lx < P.wx && P.ly < P.wy && P.lz < P.wz;
  const int ax = P.act ? P.lx : 0, ay = P.act ? P.ly : 0, az = P.act ? P.lz : 0;
  P.v = (unsigned)(P.ox + ax) + (unsigned)g.nx * ((unsigned)(P.oy + ay) + (unsigned)g.ny * (unsigned)(P.oz + az));
  return P;
}

// u of the brick and its halo into LDS (zero without uin). Positions past a
// cut brick's halo repeat its last ones: no active pair reads them.
template <int NR>
__device__ __forceinline__ void st_stage_u(const Geom& g, const StPair& P, const float* __restrict__ uin,
                                           float (*su)[kHalo * kStPlane]) {
  constexpr int kH3 = kHalo * kHalo * kHalo;
  constexpr int kTrips = (kH3 + kStBrickThreads - 1) / kStBrickThreads;
  const int t = threadIdx.x;
  if (!uin) {
    float* z = su[0];
    for (int i = t; i < NR * kHalo * kStPlane; i += kStBrickThreads) z[i] = 0.f;
    return;
  }
  float hv[kTrips][NR];
#pragma unroll
  for (int r = 0; r < kTrips; r++) {
    const int i = min(t + kStBrickThreads * r, kH3 - 1);
    const int hx = min(i % kHalo, P.wx + 1), hy = min((i / kHalo) % kHalo, P.wy + 1),
              hz = min(i / (kHalo * kHalo), P.wz + 1);
    const unsigned w = (unsigned)wrapm(P.ox + hx - 1, g.nx) +
                       (unsigned)g.nx * ((unsigned)wrapm(P.oy + hy - 1, g.ny) +
                                         (unsigned)g.ny * (unsigned)wrapm(P.oz + hz - 1, g.nz));
#pragma unroll
    for (int k = 0; k < NR; k++) hv[r][k] = ld_off(uin + (size_t)k * (size_t)g.nn, 4u * w);
  }
#pragma unroll
  for (int r = 0; r < kTrips; r++) {
    const int i = t + kStBrickThreads * r;
    const int hx = i % kHalo, hy = (i / kHalo) % kHalo, hz = i / (kHalo * kHalo);
    if (i < kH3) {
#pragma unroll
      for (int k = 0; k < NR; k++) su[k][hx + kStPitch * hy + kStPlane * hz] = hv[r][k];
    }
  }
}

// A pair's couplings (first node a, second b) and diagonals. FP16 couplings
// stay divided by the level's scale, which the sums are multiplied with;
// they are held packed (kStPacked), half the registers for multiply-adds at
// half the rate, or widened (kStWide): the same values and bits.
enum StForm : int { kStFp32 = 0, kStPacked = 1, kStWide = 2 };
template <int FORM>
struct StCoef {
  f32x2 c[27];
  float scale;
  __device__ __forceinline__ void load(const StRef& S, size_t nn, unsigned v) {
    if constexpr (FORM == kStFp32) {
#pragma unroll
      for (int o = 0; o < 27; o++) c[o] = *(const f32x2*)((const char*)(S.f32 + o * nn) + 4u * v);
    } else {
      scale = *S.scale;
      f32x2 off = {0.f, 0.f};
#pragma unroll
      for (int o = 0; o < 27; o++) {
        if (o == 13) continue;
        const f16x2 h = *(const f16x2*)((const char*)(S.f16 + o * nn) + 2u * v);
        c[o] = f32x2{(float)h.x, (float)h.y};
        off.x += c[o].x;
        off.y += c[o].y;
      }
      c[13] = f32x2{-off.x * scale, -off.y * scale};  // minus the sum of the couplings
    }
  }
  __device__ __forceinline__ f32x2 diag() const { return c[13]; }
  __device__ __forceinline__ float scaled(float s) const { return FORM == kStFp32 ? s : s * scale; }
  __device__ __forceinline__ float fma_a(int o, float w, float s) const { return fmaf(c[o].x, w, s); }
  __device__ __forceinline__ float fma_b(int o, float w, float s) const { return fmaf(c[o].y, w, s); }
};
template <>
struct StCoef<kStPacked> {
  f16x2 c[27];
  float scale;
  __device__ __forceinline__ void load(const StRef& S, size_t nn, unsigned v) {
    scale = *S.scale;
#pragma unroll
    for (int o = 0; o < 27; o++)
      if (o != 13) c[o] = *(const f16x2*)((const char*)(S.f16 + o * nn) + 2u * v);
  }
  __device__ __forceinline__ f32x2 diag() const {
    f32x2 off = {0.f, 0.f};
#pragma unroll
    for (int o = 0; o < 27; o++)
      if (o != 13) {
        off.x += (float)c[o].x;
        off.y += (float)c[o].y;
      }
    return f32x2{-off.x * scale, -off.y * scale};
  }
  __device__ __forceinline__ float scaled(float s) const { return s * scale; }
  // Takes either half of the packed register as it is. (Written as fmaf of
  // a widened value, the compiler widens all couplings ahead of the sweeps.)
  __device__ __forceinline__ float fma_a(int o, float w, float s) const {
    asm("v_fma_mix_f32 %0, %1, %2, %0 op_sel_hi:[1,0,0]" : "+v"(s) : "v"(c[o]), "v"(w));
    return s;
  }
  __device__ __forceinline__ float fma_b(int o, float w, float s) const {
    asm("v_fma_mix_f32 %0, %1, %2, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(s) : "v"(c[o]), "v"(w));
    return s;
  }
};

// Sums of the pair's couplings to the eight rows other than its own, with
// the reads of two rows in flight (left to itself the compiler issues all of
// them first, for 150 registers and a third of the resident workgroups).
template <int NR, class Coef>
__device__ __forceinline__ void st_other_rows(const Coef& C, const float (*su)[kHalo * kStPlane], int base,
                                              float (&sa)[NR], float (&sb)[NR]) {
  f32x2 w[3][NR][2];
  auto fetch = [&](int i) {
    const int r = i < 4 ? i : i + 1, off = base + kStPitch * (r % 3 - 1) + kStPlane * (r / 3 - 1);
#pragma unroll
    for (int k = 0; k < NR; k++) {
      w[i % 3][k][0] = *(const f32x2*)&su[k][off];
      w[i % 3][k][1] = *(const f32x2*)&su[k][off + 2];
    }
  };
#pragma unroll
  for (int k = 0; k < NR; k++) sa[k] = sb[k] = 0.f;
  fetch(0);
  fetch(1);
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int r = i < 4 ? i : i + 1;
    if (i + 2 < 8) fetch(i + 2);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < NR; k++) {
      const f32x2 w01 = w[i % 3][k][0], w23 = w[i % 3][k][1];
      sa[k] = C.fma_a(3 * r, w01.x, sa[k]);
      sb[k] = C.fma_b(3 * r, w01.y, sb[k]);
      sa[k] = C.fma_a(3 * r + 1, w01.y, sa[k]);
      sb[k] = C.fma_b(3 * r + 1, w23.x, sb[k]);
      sa[k] = C.fma_a(3 * r + 2, w23.x, sa[k]);
      sb[k] = C.fma_b(3 * r + 2, w23.y, sb[k]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Value of the next / previous lane of a row of 16.
__device__ __forceinline__ float row_next(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x101, 0xF, 0xF, true));
}
__device__ __forceinline__ float row_prev(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x111, 0xF, 0xF, true));
}

template <bool FORWARD, int NR, class Coef>
__device__ __forceinline__ void st_brick_sweeps(const StPair& P, const Coef& C, float (*su)[kHalo * kStPlane],
                                                const f32x2 (&fv)[NR], f32x2 inv, int sweeps,
                                                f32x2 (&u)[NR]) {
  const int w = (int)threadIdx.x >> 6;
  const int base = P.lx + kStPitch * (P.ly + 1) + kStPlane * (P.lz + 1);  // the node before the pair
  const bool has_prev = P.lx > 0, has_next = P.lx + 2 < P.wx;
#pragma unroll 1
  for (int s = 0; s < 4 * sweeps; s++) {
    const int p = FORWARD ? (s & 3) : 3 - (s & 3);
    if (w == p) {
      float sa[NR], sb[NR];
      st_other_rows<NR>(C, su, base, sa, sb);
#pragma unroll
      for (int k = 0; k < NR; k++) {
        const f32x2 w01 = *(const f32x2*)&su[k][base], w23 = *(const f32x2*)&su[k][base + 2];
        if (FORWARD) {
          sa[k] = C.fma_a(12, w01.x, C.fma_a(14, w23.x, sa[k]));
          u[k].x = (fv[k].x - C.scaled(sa[k])) * inv.x;
          const float nx = row_next(u[k].x);
          sb[k] = C.fma_b(12, u[k].x, C.fma_b(14, has_next ? nx : w23.y, sb[k]));
          u[k].y = (fv[k].y - C.scaled(sb[k])) * inv.y;
        } else {
          sb[k] = C.fma_b(12, w01.y, C.fma_b(14, w23.y, sb[k]));
          u[k].y = (fv[k].y - C.scaled(sb[k])) * inv.y;
          const float pv = row_prev(u[k].y);
          sa[k] = C.fma_a(12, has_prev ? pv : w01.x, C.fma_a(14, u[k].y, sa[k]));
          u[k].x = (fv[k].x - C.scaled(sa[k])) * inv.x;
        }
        if (P.act) {
          su[k][base + 1] = u[k].x;
          su[k][base + 2] = u[k].y;
        }
      }
    }
    __syncthreads();
  }
}

// NR load cases from k0 on of block b's brick.
template <int FORM, int NR>
__device__ inline void st_brick_body(const Geom& g, const StRef& S, const float* __restrict__ f,
                                     const float* __restrict__ uin, float* __restrict__ uout, int sweeps, int forward,
                                     int zero_in, int b, int k0) {
  auto& su = st_brick_lds().su;
  const StPair P = st_pair(g, b);
  const size_t nn = (size_t)g.nn;
  StCoef<FORM> C;
  C.load(S, nn, P.v);
  f32x2 fv[NR], u[NR];
#pragma unroll
  for (int k = 0; k < NR; k++) fv[k] = *(const f32x2*)((const char*)(f + (k0 + k) * nn) + 4u * P.v);
  st_stage_u<NR>(g, P, zero_in ? nullptr : uin + k0 * nn, su);
  const f32x2 dg = C.diag(), inv = {1.f / dg.x, 1.f / dg.y};
  __syncthreads();
  if (forward)
    st_brick_sweeps<true, NR>(P, C, su, fv, inv, sweeps, u);
  else
    st_brick_sweeps<false, NR>(P, C, su, fv, inv, sweeps, u);
  if (P.act) {
#pragma unroll
    for (int k = 0; k < NR; k++) *(f32x2*)((char*)(uout + (k0 + k) * nn) + 4u * P.v) = u[k];
  }
}

// ---- setup bodies (Galerkin hierarchy, FP16 packing, coarsest inverse) ----
// Level-1 element matrices from kappa: E(E) = sum_c kappa_c G[c].
__device__ inline void galerkin_first_body(const Geom& fg, const Geom& cg, const GalerkinConsts& G,
                                           const float* __restrict__ kappa, float* __restrict__ E, long long t) {
  if (t >= cg.nn) return;
  int X, Y, Z;
  split_node(cg.nx, cg.ny, t, X, Y, Z);
  float kc[8];
#pragma unroll
  for (int c = 0; c < 8; c++)
    kc[c] = kappa[lin(fg, 2 * X + (c & 1), 2 * Y + ((c >> 1) & 1), 2 * Z + (c >> 2))];
#pragma unroll
  for (int q = 0; q < 36; q++) {
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < 8; c++) s += kc[c] * G.G[c][q];
    E[q * cg.nn + t] = s;
  }
}

// 1-D interpolation weight of a fine point p (0..2) from coarse corner M (0/1).
__device__ constexpr float w1d(int p, int M) {
  return (p - 2 * M == 0) ? 1.f : ((p - 2 * M == 1 || p - 2 * M == -1) ? 0.5f : 0.f);
}

// Deeper levels: Eout(E) = sum_c Q_c^T Ein(child c) Q_c.
__device__ inline void galerkin_next_body(const Geom& fg, const Geom& cg, const float* __restrict__ Ein,
                                          float* __restrict__ Eout, long long t) {
  if (t >= cg.nn) return;
  int X, Y, Z;
  split_node(cg.nx, cg.ny, t, X, Y, Z);
  float acc[36];
#pragma unroll
  for (int q = 0; q < 36; q++) acc[q] = 0.f;
#pragma unroll
  for (int c = 0; c < 8; c++) {
    const int cx = c & 1, cy = (c >> 1) & 1, cz = c >> 2;
    const long long child = lin(fg, 2 * X + cx, 2 * Y + cy, 2 * Z + cz);
    float e[36];
#pragma unroll
    for (int q = 0; q < 36; q++) e[q] = Ein[q * fg.nn + child];
    // T = E Q  (8 x 8)
    float T[8][8];
#pragma unroll
    for (int m = 0; m < 8; m++)
#pragma unroll
      for (int b = 0; b < 8; b++) {
        float s = 0.f;
#pragma unroll
        for (int n = 0; n < 8; n++) {
          const float qnb = w1d(cx + (n & 1), b & 1) * w1d(cy + ((n >> 1) & 1), (b >> 1) & 1) *
                            w1d(cz + (n >> 2), b >> 2);
          if (qnb != 0.f) s += e[tri8(m, n)] * qnb;
        }
        T[m][b] = s;
      }
    // acc(a,b) += sum_m Q(m,a) T(m,b)
#pragma unroll
    for (int a = 0; a < 8; a++)
#pragma unroll
      for (int b = a; b < 8; b++) {
        float s = 0.f;
#pragma unroll
        for (int m = 0; m < 8; m++) {
          const float qma = w1d(cx + (m & 1), a & 1) * w1d(cy + ((m >> 1) & 1), (a >> 1) & 1) *
                            w1d(cz + (m >> 2), a >> 2);
          if (qma != 0.f) s += qma * T[m][b];
        }
        acc[tri8(a, b)] += s;
      }
  }
#pragma unroll
  for (int q = 0; q < 36; q++) Eout[q * cg.nn + t] = acc[q];
}

// Node stencil from element matrices; the diagonal is reset to minus the sum
// of the off-diagonal couplings so that constants stay in the null space.
__device__ inline void stencil_from_elements_body(const Geom& g, const float* __restrict__ E, float* __restrict__ st,
                                                  long long t) {
  if (t >= g.nn) return;
  int x, y, z;
  split_node(g.nx, g.ny, t, x, y, z);
  float a[27];
#pragma unroll
  for (int o = 0; o < 27; o++) a[o] = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const int ax = e & 1, ay = (e >> 1) & 1, az = e >> 2;
    const int ex = wrapm(x - 1 + ax, g.nx), ey = wrapm(y - 1 + ay, g.ny), ez = wrapm(z - 1 + az, g.nz);
    const long long eid = lin(g, ex, ey, ez);
    const int lv = (1 - ax) + 2 * (1 - ay) + 4 * (1 - az);
#pragma unroll
    for (int m = 0; m < 8; m++) {
      const int o = (ax + (m & 1)) + 3 * (ay + ((m >> 1) & 1)) + 9 * (az + (m >> 2));
      a[o] += E[tri8(lv, m) * g.nn + eid];
    }
  }
  double off = 0.0;
#pragma unroll
  for (int o = 0; o < 27; o++)
    if (o != 13) off += (double)a[o];
  a[13] = (float)(-off);
#pragma unroll
  for (int o = 0; o < 27; o++) st[o * g.nn + t] = a[o];
}

// Largest |coupling| of a level (as float bits: non-negative floats order
// like their bit patterns), for the FP16 scale; block lb of nb.
__device__ inline void stencil_absmax_body(const Geom& g, const float* __restrict__ st, unsigned int* __restrict__ bits,
                                           int lb, int nb) {
  float m = 0.f;
  for (long long v = (long long)lb * blockDim.x + threadIdx.x; v < g.nn; v += (long long)nb * blockDim.x)
#pragma unroll
    for (int o = 0; o < 27; o++)
      if (o != 13) m = fmaxf(m, fabsf(st[o * g.nn + v]));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_down(m, o, 64));
  __shared__ float wm[kWaves];
  if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kWaves; w++) m = fmaxf(m, wm[w]);
    atomicMax(bits, __float_as_uint(m));
  }
}

// FP16 copy of a level's couplings divided by the level scale. Coupling
// (v, v+d) for d before the centre in offset order is taken from the
// neighbour's entry (v+d, v), so the stored operator is exactly symmetric.
__device__ inline void stencil_pack_body(const Geom& g, const float* __restrict__ st, const float* __restrict__ scale,
                                         _Float16* __restrict__ st16, long long t) {
  if (t >= g.nn) return;
  int x, y, z;
  split_node(g.nx, g.ny, t, x, y, z);
  const float sc = *scale;
  const float inv = sc > 0.f ? 1.f / sc : 0.f;
#pragma unroll
  for (int o = 0; o < 27; o++) {
    float val = 0.f;
    if (o > 13) {
      val = st[o * g.nn + t];
    } else if (o < 13) {
      const long long w = lin(g, wrapm(x + o % 3 - 1, g.nx), wrapm(y + (o / 3) % 3 - 1, g.ny),
                              wrapm(z + o / 9 - 1, g.nz));
      val = st[(26 - o) * g.nn + w];
    }
    st16[o * g.nn + t] = (_Float16)(val * inv);
  }
}

// Coarsest level: dense FP64 matrix from the stencil, symmetrised, zero row
// sums, plus (tr/n^2) * 1 1^T to remove the constant null space (the
// reference solves its coarsest system on the host with Eigen and a
// null-space projection, grid.cpp:272-310, :432-510). The result is its
// explicit inverse Binv, so every V-cycle's coarsest solve is one small
// dense matrix-vector product on the device.
//
// The inverse is a blocked Gauss-Jordan elimination of the SPD matrix (no
// pivoting), kGjB pivots per step, K the step's pivot rows, O all others:
//   D = A_KK^-1,  A_KK <- D,  A_KO <- D A_KO,  A_OK <- -A_OK D,
//   A_OO <- A_OO - A_OK (D A_KO),
// the products in FP64 matrix instructions. With the columns of K in the
// old pivot rows replaced by the identity and the old A_OK by zero, all four
// are one rule: R = D A_K:, rows of K become R, other rows A - A_:K R.
constexpr int kGjB = 32;            // pivots per step
constexpr int kGjTile = 64;         // tile edge of a workgroup
constexpr int kInvertLdsMax = 64;   // one workgroup holds the matrix in LDS up to this size

// Row strides (doubles) of the LDS operands: 16 rows 34 apart, and two rows
// 80 apart, start on different banks.
constexpr int kGjStrideC = kGjB + 2, kGjStrideR = kGjTile + 16;

typedef double f64x4 __attribute__((ext_vector_type(4)));

// Entry (i, j), i != j, of the symmetrised coarse matrix: the mean of the
// two stencil entries that describe the coupling (a coarsest edge has at
// least 3 nodes, so there is one pair), 0 between nodes that do not touch.
// ci and cj are the nodes' coordinates packed by gj_coord.
__device__ inline int gj_coord(const Geom& g, int i) {
  int x, y, z;
  split_node(g.nx, g.ny, i, x, y, z);
  return x | (y << 10) | (z << 20);
}
__device__ inline double gj_offdiag(const Geom& g, const float* __restrict__ st, int i, int ci, int j, int cj) {
  const int n = (int)g.nn;
  const int dims[3] = {g.nx, g.ny, g.nz};
  int o = 0, w = 1;
  bool touch = true;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    int d = ((cj >> (10 * a)) & 1023) - ((ci >> (10 * a)) & 1023);
    if (d == dims[a] - 1) d = -1;
    else if (d == 1 - dims[a]) d = 1;
    touch = touch && d >= -1 && d <= 1;
    o += w * (d + 1);
    w *= 3;
  }
  o = touch ? o : 13;  // loads without a branch, so several entries' are in flight
  const double a = 0.5 * ((double)st[o * n + i] + (double)st[(26 - o) * n + j]);
  return touch ? a : 0.0;
}

// Minus the sum of node v's off-diagonal couplings, by 32 lanes (every lane
// gets it).
__device__ inline double gj_diag(const Geom& g, const float* __restrict__ st, int v) {
  const int n = (int)g.nn, o = (int)threadIdx.x & 31;
  double a = 0.0;
  if (o < 27 && o != 13) {
    int x, y, z;
    split_node(g.nx, g.ny, v, x, y, z);
    const int w = wrapm(x + o % 3 - 1, g.nx) +
                  g.nx * (wrapm(y + (o / 3) % 3 - 1, g.ny) + g.ny * wrapm(z + o / 9 - 1, g.nz));
    a = 0.5 * ((double)st[o * n + v] + (double)st[(26 - o) * n + w]);
  }
#pragma unroll
  for (int m = 16; m > 0; m >>= 1) a += __shfl_xor(a, m, 64);
  return -a;
}

// 1/v of a pivot (finite, positive): the hardware estimate and two
// Newton-Raphson steps, within an ulp.
__device__ inline double gj_rcp(double v) {
  double r = __builtin_amdgcn_rcp(v);
  r = fma(fma(-v, r, 1.0), r, r);
  r = fma(fma(-v, r, 1.0), r, r);
  return r;
}

// In-place inverse of the kGjB x kGjB SPD matrix m (LDS, row stride
// kGjStrideC) by 256 threads: thread t keeps rows 4 (t/32) .. + 3 of column
// t%32 in registers. Blocked Gauss-Jordan with four pivots a step: the 32
// threads that own the pivot rows write them to LDS, one barrier, and every
// thread factors the 4 x 4 pivot block (L D L^T, the scalar elimination's
// arithmetic) and solves for its column. The elimination keeps the matrix
// symmetric up to the sign between eliminated and remaining indices, so the
// pivot columns come from the same rows. Bound by its serial chain, 8 steps
// of one barrier and four reciprocals each: about 8 us. One pivot a step (32
// barriers) took 13 us; the matrix in LDS, two barriers, a division and
// runtime index divisions a step 29 us.
constexpr int kGjP = 4;  // pivots of such a step
__device__ __forceinline__ void gj_invert_block(double* m, double (*rows)[kGjP][kGjB]) {
  const int j = (int)threadIdx.x & 31, ib = (int)threadIdx.x >> 5, i0 = kGjP * ib;
  double a[kGjP];
#pragma unroll
  for (int r = 0; r < kGjP; r++) a[r] = m[(i0 + r) * kGjStrideC + j];
#pragma unroll 1  // one step's code stays in the instruction cache
  for (int s = 0; s < kGjB / kGjP; s++) {
    double(*X)[kGjB] = rows[s & 1];
    if (ib == s) {
#pragma unroll
      for (int r = 0; r < kGjP; r++) X[r][j] = a[r];
    }
    __syncthreads();
    const int k0 = kGjP * s;
    double P[kGjP][kGjP], L[kGjP][kGjP], d[kGjP], t[kGjP];
#pragma unroll
    for (int u = 0; u < kGjP; u++) {
#pragma unroll
      for (int v = 0; v < kGjP; v++) P[u][v] = X[u][k0 + v];
      t[u] = X[u][j];
    }
    const bool inK = j >= k0 && j < k0 + kGjP;
#pragma unroll
    for (int u = 0; u < kGjP; u++)
      if (inK) t[u] = j == k0 + u ? 1.0 : 0.0;
#pragma unroll
    for (int u = 0; u < kGjP; u++) {
      d[u] = gj_rcp(P[u][u]);
#pragma unroll
      for (int v = u + 1; v < kGjP; v++) {
        L[v][u] = P[u][v] * d[u];
#pragma unroll
        for (int w = u + 1; w <= v; w++) P[w][v] = fma(-L[v][u], P[u][w], P[w][v]);
        t[v] = fma(-L[v][u], t[u], t[v]);
      }
    }
#pragma unroll
    for (int u = kGjP - 1; u >= 0; u--) {
      t[u] *= d[u];
#pragma unroll
      for (int v = u + 1; v < kGjP; v++) t[u] = fma(-L[v][u], t[v], t[u]);
    }
    const double sign = ib < s ? 1.0 : -1.0;  // minus the pivot columns' entries
#pragma unroll
    for (int r = 0; r < kGjP; r++) {
      double v = inK ? 0.0 : a[r];
#pragma unroll
      for (int u = 0; u < kGjP; u++) v = fma(sign * X[u][i0 + r], t[u], v);
      a[r] = ib == s ? t[r] : v;
    }
  }
#pragma unroll
  for (int r = 0; r < kGjP; r++) m[(i0 + r) * kGjStrideC + j] = a[r];
  __syncthreads();
}

// One 16 x 16 tile of A B over kGjB terms: A rows (stride sa) and B columns
// (stride sb) start at a and b. Lane l holds A[l%16][4q + l/16] and
// B[4q + l/16][l%16] of each instruction, and results (4r + l/16, l%16).
__device__ __forceinline__ f64x4 gj_mma(const double* a, int sa, const double* b, int sb, f64x4 acc) {
  const int l = (int)threadIdx.x & 63, lr = l & 15, lk = l >> 4;
#pragma unroll
  for (int q = 0; q < kGjB / 4; q++)
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[lr * sa + 4 * q + lk], b[(4 * q + lk) * sb + lr], acc, 0, 0, 0);
  return acc;
}

// n <= kInvertLdsMax: one workgroup, the matrix in LDS. Each wave owns 16
// rows, so after the barrier behind R a step updates them in place. At n =
// 64, two steps, 29 us; the scalar elimination in LDS, two barriers a pivot,
// took 67 us (n = 125: 230 us; now four launches of 11 us).
struct GjSmallLds {
  double A[kGjTile * kGjStrideR];
  double R[kGjB * kGjStrideR];
  double D[kGjB * kGjStrideC];
  double rows[2][kGjP][kGjB];
  double diag[kGjTile];
  int coord[kGjTile];
};
__device__ inline void coarsest_invert_small_body(const Geom& g, const float* __restrict__ st,
                                                  double* __restrict__ Binv) {
  __shared__ GjSmallLds S;
  const int n = (int)g.nn, tid = threadIdx.x, l = tid & 63, w = tid >> 6;
  if (tid < kGjTile) {
    S.coord[tid] = tid < n ? gj_coord(g, tid) : 0;
    S.diag[tid] = 0.0;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kGjTile * 32 / kBlock; r++) {
    const int v = (tid >> 5) + (kBlock / 32) * r;
    const double d = gj_diag(g, st, min(v, n - 1));
    if ((tid & 31) == 0 && v < n) S.diag[v] = d;
  }
  __syncthreads();
  const double alpha = wave_sum(S.diag[l]) / ((double)n * (double)n);
  // padded with the identity beyond n
#pragma unroll 4
  for (int q = tid; q < kGjTile * kGjTile; q += kBlock) {
    const int i = q / kGjTile, j = q % kGjTile;
    const double o = gj_offdiag(g, st, min(i, n - 1), S.coord[i], min(j, n - 1), S.coord[j]);
    S.A[i * kGjStrideR + j] = (i < n && j < n) ? (i == j ? S.diag[i] : o) + alpha : (i == j ? 1.0 : 0.0);
  }
  __syncthreads();
  for (int k0 = 0; k0 < n; k0 += kGjB) {
    for (int q = tid; q < kGjB * kGjB; q += kBlock)
      S.D[(q / kGjB) * kGjStrideC + q % kGjB] = S.A[(k0 + q / kGjB) * kGjStrideR + k0 + q % kGjB];
    __syncthreads();
    gj_invert_block(S.D, S.rows);
    // the pivot rows with the identity in the columns of K
    for (int q = tid; q < kGjB * kGjB; q += kBlock)
      S.A[(k0 + q / kGjB) * kGjStrideR + k0 + q % kGjB] = q / kGjB == q % kGjB ? 1.0 : 0.0;
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const f64x4 r = gj_mma(S.D + 16 * h * kGjStrideC, kGjStrideC, S.A + k0 * kGjStrideR + 16 * w, kGjStrideR,
                             f64x4{0, 0, 0, 0});
#pragma unroll
      for (int q = 0; q < 4; q++) S.R[(16 * h + 4 * q + (l >> 4)) * kGjStrideR + 16 * w + (l & 15)] = r[q];
    }
    __syncthreads();
    const bool pivot = 16 * w >= k0 && 16 * w < k0 + kGjB;  // this wave's rows are pivot rows
    f64x4 out[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const f64x4 acc = gj_mma(S.A + 16 * w * kGjStrideR + k0, kGjStrideR, S.R + 16 * c, kGjStrideR, f64x4{0, 0, 0, 0});
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int i = 16 * w + 4 * q + (l >> 4), j = 16 * c + (l & 15);
        const bool inK = j >= k0 && j < k0 + kGjB;
        out[c][q] = pivot ? S.R[(i - k0) * kGjStrideR + j] : (inK ? 0.0 : S.A[i * kGjStrideR + j]) - acc[q];
      }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int q = 0; q < 4; q++) S.A[(16 * w + 4 * q + (l >> 4)) * kGjStrideR + 16 * c + (l & 15)] = out[c][q];
    __syncthreads();
  }
  for (int q = tid; q < n * n; q += kBlock) {
    const int i = q / n, j = q - i * n;
    Binv[q] = 0.5 * (S.A[i * kGjStrideR + j] + S.A[j * kGjStrideR + i]);
  }
}

// Larger n: every step is one launch over kGjTile x kGjTile tiles. The step
// reads one n x n matrix and writes another (every entry changes anyway), so
// its workgroups need no order among them, and each forms the R columns of
// its own tile; the workgroup whose tile holds the next pivot block inverts
// that block right away, and so the serial part runs beside the other tiles.
// A step is bound by that chain: 11.3 us at n = 216 and 576, 15.6 us at 1331
// (three launches a step with the 29 us inverse on its own: 51, 53 and 59 us;
// the whole inverse 370, 1000 and 2500 us before, 100, 230 and 690 us now).
// Work space of a level: the second n x n matrix, two pivot inverses, the
// diagonal. The matrices are work and Binv by turns, the last result in work.
__host__ __device__ inline long long gj_tiles(const Geom& g) { return (g.nn + kGjTile - 1) / kGjTile; }
__host__ __device__ inline int gj_steps(const Geom& g) { return (int)((g.nn + kGjB - 1) / kGjB); }
struct GjWork {
  double *even, *odd;  // the matrix before even / odd steps
  double* D[2];        // pivot inverse of even / odd steps
  double* diag;
};
__host__ __device__ inline GjWork gj_work(const Geom& g, double* work, double* Binv) {
  GjWork W;
  const bool last_even = (gj_steps(g) & 1) == 0;  // the result is in `even`
  W.even = last_even ? work : Binv;
  W.odd = last_even ? Binv : work;
  W.D[0] = work + g.nn * g.nn;
  W.D[1] = W.D[0] + kGjB * kGjB;
  W.diag = W.D[1] + kGjB * kGjB;
  return W;
}

// Diagonal, 32 lanes per node (8 nodes per block).
__device__ inline void gj_diag_body(const Geom& g, const float* __restrict__ st, const GjWork& W, int lb) {
  const int v = lb * (kBlock / 32) + ((int)threadIdx.x >> 5);
  if (v >= (int)g.nn) return;
  const double d = gj_diag(g, st, v);
  if ((threadIdx.x & 31) == 0) W.diag[v] = d;
}

struct GjLds {
  double X[kGjB * kGjStrideR];     // old pivot rows of the tile's columns
  double R[kGjB * kGjStrideR];     // D X
  double C[kGjTile * kGjStrideC];  // old pivot columns of the tile's rows
  double D[kGjB * kGjStrideC];     // pivot inverse; then the next pivot block
  double rows[2][kGjP][kGjB];
};
__device__ inline GjLds& gj_lds() {
  __shared__ GjLds lds;
  return lds;
}

// Inverts the pivot block of step s that the workgroup has put in lds.D
// (identity beyond n) and publishes it for the step.
__device__ inline void gj_publish_pivot(const GjWork& W, int s) {
  GjLds& L = gj_lds();
  __syncthreads();
  gj_invert_block(L.D, L.rows);
  for (int q = threadIdx.x; q < kGjB * kGjB; q += kBlock)
    W.D[s & 1][q] = L.D[(q / kGjB) * kGjStrideC + q % kGjB];
}

// Tile lb of the matrix, with alpha = tr / n^2 on every entry; the first
// tile also inverts the first pivot block.
__device__ inline void gj_assemble_body(const Geom& g, const float* __restrict__ st, const GjWork& W, int lb) {
  GjLds& L = gj_lds();
  __shared__ int coord[2][kGjTile];
  __shared__ double sh[kWaves], alpha_sh;
  const int n = (int)g.nn, nt = (int)gj_tiles(g), tid = threadIdx.x;
  const int i0 = (lb / nt) * kGjTile, j0 = (lb % nt) * kGjTile;
  if (tid < 2 * kGjTile) {
    const int h = tid / kGjTile, v = (h ? j0 : i0) + tid % kGjTile;
    coord[h][tid % kGjTile] = v < n ? gj_coord(g, v) : 0;
  }
  double tr[1] = {0.0};
  for (int i = tid; i < n; i += kBlock) tr[0] += W.diag[i];
  block_sum<1>(tr, sh);
  if (tid == 0) alpha_sh = tr[0] / ((double)n * (double)n);
  __syncthreads();
  const double alpha = alpha_sh;
#pragma unroll 4
  for (int q = tid; q < kGjTile * kGjTile; q += kBlock) {
    const int a = q / kGjTile, b = q % kGjTile, i = i0 + a, j = j0 + b;
    const int ic = min(i, n - 1), jc = min(j, n - 1);
    const double o = gj_offdiag(g, st, ic, coord[0][a], jc, coord[1][b]), dg = W.diag[ic];
    const double v = (i < n && j < n) ? (i == j ? dg : o) + alpha : (i == j ? 1.0 : 0.0);
    if (i < n && j < n) W.even[(long long)i * n + j] = v;
    if (lb == 0 && a < kGjB && b < kGjB) L.D[a * kGjStrideC + b] = v;
  }
  if (lb == 0) gj_publish_pivot(W, 0);
}

// Tile lb of elimination step s.
__device__ inline void gj_step_body(const Geom& g, const GjWork& W, int s, int lb) {
  GjLds& L = gj_lds();
  const int n = (int)g.nn, nt = (int)gj_tiles(g), tid = threadIdx.x, l = tid & 63, w = tid >> 6;
  const int i0 = (lb / nt) * kGjTile, j0 = (lb % nt) * kGjTile, k0 = s * kGjB;
  const double* __restrict__ src = (s & 1) ? W.odd : W.even;
  double* __restrict__ dst = (s & 1) ? W.even : W.odd;
  const double* __restrict__ D = W.D[s & 1];
  // All loads of the tile in flight together, from clamped positions, before
  // the first LDS store; entries beyond n become zero (and the identity in
  // the columns of K) on the way. As guarded loads they waited for each
  // other.
  constexpr int kXT = kGjB * kGjTile / kBlock, kDT = kGjB * kGjB / kBlock;
  double old[4][4], xv[kXT], cv[kXT], dv[kDT];
#pragma unroll
  for (int t = 0; t < kDT; t++) dv[t] = D[tid + kBlock * t];
#pragma unroll
  for (int t = 0; t < kXT; t++) {
    const int q = tid + kBlock * t;
    const int k = min(k0 + q / kGjTile, n - 1), j = min(j0 + q % kGjTile, n - 1);
    xv[t] = src[(long long)k * n + j];
    const int i = min(i0 + q / kGjB, n - 1), c = min(k0 + q % kGjB, n - 1);
    cv[t] = src[(long long)i * n + c];
  }
#pragma unroll
  for (int c = 0; c < 4; c++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int i = i0 + 16 * w + 4 * q + (l >> 4), j = j0 + 16 * c + (l & 15);
      old[c][q] = src[(long long)min(i, n - 1) * n + min(j, n - 1)];
    }
#pragma unroll
  for (int t = 0; t < kDT; t++) {
    const int q = tid + kBlock * t;
    L.D[(q / kGjB) * kGjStrideC + q % kGjB] = dv[t];
  }
#pragma unroll
  for (int t = 0; t < kXT; t++) {
    const int q = tid + kBlock * t;
    const int k = k0 + q / kGjTile, j = j0 + q % kGjTile;
    const bool inK = j >= k0 && j < k0 + kGjB;
    L.X[(q / kGjTile) * kGjStrideR + q % kGjTile] = inK ? (j == k ? 1.0 : 0.0) : ((k < n && j < n) ? xv[t] : 0.0);
    const int i = i0 + q / kGjB, c = k0 + q % kGjB;
    L.C[(q / kGjB) * kGjStrideC + q % kGjB] = (i < n && c < n) ? cv[t] : 0.0;
  }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const f64x4 r = gj_mma(L.D + 16 * h * kGjStrideC, kGjStrideC, L.X + 16 * w, kGjStrideR, f64x4{0, 0, 0, 0});
#pragma unroll
    for (int q = 0; q < 4; q++) L.R[(16 * h + 4 * q + (l >> 4)) * kGjStrideR + 16 * w + (l & 15)] = r[q];
  }
  __syncthreads();
  // k1: the next pivot block, when this tile holds it
  const int k1 = k0 + kGjB;
  const bool next = k1 < n && i0 == j0 && k1 >= i0 && k1 < i0 + kGjTile;
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const f64x4 acc = gj_mma(L.C + 16 * w * kGjStrideC, kGjStrideC, L.R + 16 * c, kGjStrideR, f64x4{0, 0, 0, 0});
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int a = 16 * w + 4 * q + (l >> 4), b = 16 * c + (l & 15), i = i0 + a, j = j0 + b;
      const bool pivot = i >= k0 && i < k0 + kGjB;
      const bool inK = j >= k0 && j < k0 + kGjB;
      const double v = pivot ? L.R[(i - k0) * kGjStrideR + b] : (inK ? 0.0 : old[c][q]) - acc[q];
      if (i < n && j < n) dst[(long long)i * n + j] = v;
      if (next && i >= k1 && i < k1 + kGjB && j >= k1 && j < k1 + kGjB)
        L.D[(i - k1) * kGjStrideC + j - k1] = (i < n && j < n) ? v : (i == j ? 1.0 : 0.0);
    }
  }
  if (next) gj_publish_pivot(W, s + 1);
}

// Binv from the last step's matrix, made exactly symmetric.
__device__ inline void gj_symmetrise_body(const Geom& g, const double* __restrict__ work, double* __restrict__ Binv,
                                          long long q) {
  const long long n = g.nn;
  if (q >= n * n) return;
  const long long a = q / n, b = q - a * n;
  Binv[q] = 0.5 * (work[a * n + b] + work[b * n + a]);
}

// ---- one-workgroup tail V-cycle ---------------------------------------------
// The last two levels of a hierarchy, when the first of them has at most
// kTailStartNodes nodes (8^3 and 4^3 for edges that are powers of two), are
// a few hundred nodes: as separate launches their smoothers, residual,
// transfers and coarsest product are pure launch and memory latency. One
// workgroup runs the whole V-cycle of the two: exact 8-colour Gauss-Seidel
// from zero (forward before restriction, reverse after prolongation, so the
// V-cycle stays symmetric), residual, restriction, product with the coarsest
// inverse, prolongation. A hierarchy whose coarse levels are larger has no
// tail: its coarsest level is solved by coarsest_rows_body.
//
// Bound by latency: a chain of 16 Gauss-Seidel steps at two sweeps. The work
// split is the brick smoother's for small levels (a lane owns a node pair of
// one row parity, its couplings in registers, both colours in one step),
// here one wave per row parity and load case, with the periodic neighbours
// exact: rows wrap by their offsets, an x-halo column on either side is
// written with the edge nodes. The coarsest inverse's entries are loaded
// into registers at the start, four lanes to a result. 16.4 us at 8^3 (28 us
// with 8 lanes per node, all stencils staged through LDS and 32 steps). The
// four forms share a kernel of 168 registers: the 8^3 forms need 143, the
// general ones spill (33 registers in all, 100 bytes of scratch a lane; 42
// and 112 in the batched launch).
constexpr int kTailStartNodes = 512;  // largest first tail level (8^3)
constexpr int kTailCoarseNodes = kTailStartNodes / 8;
constexpr int kTailThreads = 64 * 4 * OTM_NRHS;
constexpr int kTailTerms = kTailCoarseNodes / 4;  // coarsest product, terms of a lane
constexpr int kCoarsestMax = 4096;    // largest coarsest level
// u of one load case: rows of nx + 4, planes padded to an odd multiple of 16
// so that the reads of half a wave fall on different banks (an edge is at
// least 6, so the largest is 6 x 6 x 14)
constexpr int kTailU = 1280;
static_assert(OTM_NRHS * kTailCoarseNodes * 4 <= kTailThreads, "four lanes per coarse result");

struct TailLevels {
  int sweeps;
  Geom g, gc;          // the two levels
  StRef st;            // stencil of the first
  const float* f0;     // its right-hand side
  const double* Binv;  // inverse of the coarsest
  float* uout;         // correction of the first (output)
};

void launch_tail_vcycle(hipStream_t s, const TailLevels& T);

// This lane's pair of the tail's first level.
struct TailPair {
  int k, p;            // load case, row parity
  bool act;
  unsigned v;          // first node
  int off[9];          // LDS position of the node before the pair, per row
  int next, prev;      // lanes of the neighbouring pairs in the row
  bool first, last;    // pair at the row's begin / end
  int nx;
};

// The next / previous pair's value in the row: in a cube of 8 a row's four
// pairs are a quad of lanes.
template <bool CUBE>
__device__ __forceinline__ float tail_next(const TailPair& P, float v) {
  if constexpr (CUBE)
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x39, 0xF, 0xF, true));
  else
    return __shfl(v, P.next, 64);
}
template <bool CUBE>
__device__ __forceinline__ float tail_prev(const TailPair& P, float v) {
  if constexpr (CUBE)
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x93, 0xF, 0xF, true));
  else
    return __shfl(v, P.prev, 64);
}

template <bool FORWARD, int FORM, bool CUBE>
__device__ __forceinline__ void tail_sweeps(const TailPair& P, const StCoef<FORM>& C, float* su, f32x2 fv, f32x2 inv,
                                            int sweeps, f32x2& u) {
#pragma unroll 1
  for (int s = 0; s < 4 * sweeps; s++) {
    const int p = FORWARD ? (s & 3) : 3 - (s & 3);
    if (P.p == p) {
      float* own = su + P.off[4];
      const float o0 = own[0], o3 = own[3];
      float ra[2] = {0.f, 0.f}, rb[2] = {0.f, 0.f};  // two chains per node
#pragma unroll
      for (int r = 0; r < 9; r++) {
        if (r == 4) continue;
        const f32x2 w01 = *(const f32x2*)&su[P.off[r]], w23 = *(const f32x2*)&su[P.off[r] + 2];
        float &sa = ra[(r < 4 ? r : r - 1) & 1], &sb = rb[(r < 4 ? r : r - 1) & 1];
        sa = C.fma_a(3 * r, w01.x, sa);
        sb = C.fma_b(3 * r, w01.y, sb);
        sa = C.fma_a(3 * r + 1, w01.y, sa);
        sb = C.fma_b(3 * r + 1, w23.x, sb);
        sa = C.fma_a(3 * r + 2, w23.x, sa);
        sb = C.fma_b(3 * r + 2, w23.y, sb);
      }
      float sa = ra[0] + ra[1], sb = rb[0] + rb[1];
      if (FORWARD) {
        sa = C.fma_a(12, o0, C.fma_a(14, u.y, sa));
        u.x = (fv.x - C.scaled(sa)) * inv.x;
        sb = C.fma_b(12, u.x, C.fma_b(14, tail_next<CUBE>(P, u.x), sb));
        u.y = (fv.y - C.scaled(sb)) * inv.y;
      } else {
        sb = C.fma_b(12, u.x, C.fma_b(14, o3, sb));
        u.y = (fv.y - C.scaled(sb)) * inv.y;
        sa = C.fma_a(12, tail_prev<CUBE>(P, u.y), C.fma_a(14, u.y, sa));
        u.x = (fv.x - C.scaled(sa)) * inv.x;
      }
      if (P.act) {
        own[1] = u.x;
        own[2] = u.y;
        if (P.first) own[P.nx + 1] = u.x;
        if (P.last) own[2 - P.nx] = u.y;
      }
    }
    __syncthreads();
  }
}

// Sum over the four lanes of a quad.
__device__ __forceinline__ float quad_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false));
  return v;
}

struct alignas(16) TailLds {
  float u[OTM_NRHS][kTailU];
  float res[OTM_NRHS][kTailStartNodes];
  float fc[OTM_NRHS * kTailCoarseNodes], uc[OTM_NRHS * kTailCoarseNodes];
};
__device__ inline TailLds& tail_lds() {
  __shared__ TailLds lds;
  return lds;
}

// CUBE: 8^3 and 4^3, all index arithmetic on constants (the divisions by
// runtime edges cost 2 us).
template <int FORM, bool CUBE>
__device__ __forceinline__ void tail_form_body(const TailLevels& T) {
  TailLds& S = tail_lds();
  const Geom g = CUBE ? Geom{8, 8, 8, 512} : T.g, gc = CUBE ? Geom{4, 4, 4, 64} : T.gc;
  const int tid = threadIdx.x, m = tid & 63, w = tid >> 6;
  const int hx = g.nx >> 1, hy = g.ny >> 1, hz = g.nz >> 1, nc = (int)gc.nn;
  const int pitch = g.nx + 4, plane = ((pitch * g.ny + 15) & ~31) + 16;
  TailPair P;
  // the three waves of a parity are neighbours, so they run on three SIMDs
  P.k = w % OTM_NRHS;
  P.p = w / OTM_NRHS;
  P.act = m < hx * hy * hz;
  P.nx = g.nx;
  const int mm = P.act ? m : 0, mx = mm % hx, mr = mm / hx, my = mr % hy, mz = mr / hy;
  const int x = 2 * mx, y = 2 * my + (P.p & 1), z = 2 * mz + (P.p >> 1);
  P.v = (unsigned)(x + g.nx * (y + g.ny * z));
  P.first = mx == 0;
  P.last = mx == hx - 1;
  P.next = mm - mx + (P.last ? 0 : mx + 1);
  P.prev = mm - mx + (P.first ? hx - 1 : mx - 1);
#pragma unroll
  for (int r = 0; r < 9; r++)
    P.off[r] = x + pitch * wrapm(y + r % 3 - 1, g.ny) + plane * wrapm(z + r / 3 - 1, g.nz);
  const size_t nn = (size_t)g.nn;
  StCoef<FORM> C;
  C.load(T.st, nn, P.v);
  const f32x2 fv = *(const f32x2*)(T.f0 + P.k * nn + P.v);
  // coarse results: lane quad o = load case, node; its lanes' terms 4t + part
  const int o = tid >> 2, part = tid & 3;
  const bool has = o < OTM_NRHS * nc;
  const int ck = has ? o / nc : 0, ci = has ? o - ck * nc : 0;
  double bv[kTailTerms];
#pragma unroll
  for (int t = 0; t < kTailTerms; t++) {
    const int j = 4 * t + part;
    const double b = T.Binv[min(j, nc - 1) * nc + ci];  // symmetric
    bv[t] = j < nc ? b : 0.0;
  }
  float* su = S.u[P.k];
  for (int i = tid; i < OTM_NRHS * kTailU; i += kTailThreads) S.u[0][i] = 0.f;
  const f32x2 dg = C.diag(), inv = {1.f / dg.x, 1.f / dg.y};
  f32x2 u = {0.f, 0.f};
  __syncthreads();
  tail_sweeps<true, FORM, CUBE>(P, C, su, fv, inv, T.sweeps, u);
  {  // residual
    float sa = 0.f, sb = 0.f;
#pragma unroll
    for (int r = 0; r < 9; r++) {
      const f32x2 w01 = *(const f32x2*)&su[P.off[r]], w23 = *(const f32x2*)&su[P.off[r] + 2];
      sa = C.fma_a(3 * r, w01.x, sa);
      sb = C.fma_b(3 * r, w01.y, sb);
      if (r != 4) {
        sa = C.fma_a(3 * r + 1, w01.y, sa);
        sb = C.fma_b(3 * r + 1, w23.x, sb);
      }
      sa = C.fma_a(3 * r + 2, w23.x, sa);
      sb = C.fma_b(3 * r + 2, w23.y, sb);
    }
    if (P.act)
      *(f32x2*)&S.res[P.k][P.v] = f32x2{fv.x - fmaf(dg.x, u.x, C.scaled(sa)), fv.y - fmaf(dg.y, u.y, C.scaled(sb))};
  }
  __syncthreads();
  int cx, cy, cz;
  split_node(gc.nx, gc.ny, ci, cx, cy, cz);
  {  // restriction
    float s = 0.f;
#pragma unroll
    for (int t = 0; t < 7; t++) {
      const int q = min(4 * t + part, 26), dx = q % 3 - 1, dy = (q / 3) % 3 - 1, dz = q / 9 - 1;
      const float wt = (4 * t + part < 27 ? 1.f : 0.f) * (dx ? 0.5f : 1.f) * (dy ? 0.5f : 1.f) * (dz ? 0.5f : 1.f);
      s += wt * S.res[ck][wrapm(2 * cx + dx, g.nx) +
                          g.nx * (wrapm(2 * cy + dy, g.ny) + g.ny * wrapm(2 * cz + dz, g.nz))];
    }
    s = quad_sum(s);
    if (has && part == 0) S.fc[o] = s;
  }
  __syncthreads();
  {  // coarsest: u = Binv f, FP64 accumulation
    double s = 0.0;
#pragma unroll
    for (int t = 0; t < kTailTerms; t++) s += bv[t] * (double)S.fc[ck * nc + min(4 * t + part, nc - 1)];
    s += dpp_f64<0xB1>(s);
    s += dpp_f64<0x4E>(s);
    if (has && part == 0) S.uc[o] = (float)s;
  }
  __syncthreads();
  {  // prolongation
    const float* uc = S.uc + P.k * nc;
    const int Y1 = (y & 1) ? (my + 1 == gc.ny ? 0 : my + 1) : my, Z1 = (z & 1) ? (mz + 1 == gc.nz ? 0 : mz + 1) : mz;
    const int X1 = mx + 1 == gc.nx ? 0 : mx + 1;
    const int r00 = gc.nx * (my + gc.ny * mz), r10 = gc.nx * (Y1 + gc.ny * mz), r01 = gc.nx * (my + gc.ny * Z1),
              r11 = gc.nx * (Y1 + gc.ny * Z1);
    const float c0 = 0.25f * ((uc[r00 + mx] + uc[r10 + mx]) + (uc[r01 + mx] + uc[r11 + mx]));
    const float c1 = 0.25f * ((uc[r00 + X1] + uc[r10 + X1]) + (uc[r01 + X1] + uc[r11 + X1]));
    u.x += c0;
    u.y += 0.5f * (c0 + c1);
    if (P.act) {
      float* own = su + P.off[4];
      own[1] = u.x;
      own[2] = u.y;
      if (P.first) own[P.nx + 1] = u.x;
      if (P.last) own[2 - P.nx] = u.y;
    }
  }
  __syncthreads();
  tail_sweeps<false, FORM, CUBE>(P, C, su, fv, inv, T.sweeps, u);
  if (P.act) *(f32x2*)(T.uout + P.k * nn + P.v) = u;
}

__device__ inline void tail_vcycle_body(const TailLevels& T) {
  if (T.g.nx == 8 && T.g.ny == 8 && T.g.nz == 8) {
    if (T.st.f16)
      tail_form_body<kStWide, true>(T);
    else
      tail_form_body<kStFp32, true>(T);
  } else if (T.st.f16) {
    tail_form_body<kStWide, false>(T);
  } else {
    tail_form_body<kStFp32, false>(T);
  }
}

}  // namespace otm
