// otm_fine.hip -- single-cell launches of the matrix-free fine-level
// kernels; the device bodies are in otm_fine_dev.hpp.
#include <stdexcept>

#include "otm_fine_dev.hpp"

namespace otm {

__global__ void __launch_bounds__(kBlock) k_fine_gs_color(Geom g, FineConsts fc, const float* __restrict__ kappa,
                                                          const float* __restrict__ f, float* u, int cy, int cz) {
  fine_gs_color_body(g, fc, kappa, f, u, cy, cz, gtid());
}

__global__ void __launch_bounds__(kBlock) k_fine_residual(Geom g, FineConsts fc, const float* __restrict__ kappa,
                                                          const float* __restrict__ f, const float* __restrict__ u,
                                                          float* __restrict__ res) {
  fine_residual_body(g, fc, kappa, f, u, res, gtid());
}

__global__ void __launch_bounds__(kBlock) k_fine_apply_dot(Geom g, FineConsts fc, const float* __restrict__ kappa,
                                                           const float* __restrict__ p, float* __restrict__ q,
                                                           Reduce R) {
  fine_apply_dot_body(g, fc, kappa, p, q, R, xcd_block(), gridDim.x);
}

// LDS-tiled forms of the two (kBlock threads: BX x kBlock/BX per tile)
template <int BX>
__global__ void __launch_bounds__(kBlock) k_fine_residual_tile(Geom g, FineConsts fc, const float* __restrict__ kappa,
                                                               const float* __restrict__ f,
                                                               const float* __restrict__ u, float* __restrict__ res) {
  fine_residual_tile_body<BX, kBlock / BX>(g, fc, kappa, f, u, res, xcd_block());
}

template <int BX>
__global__ void __launch_bounds__(kBlock) k_fine_apply_tile(Geom g, FineConsts fc, const float* __restrict__ kappa,
                                                            const float* __restrict__ p, float* __restrict__ q,
                                                            Reduce R) {
  fine_apply_tile_body<BX, kBlock / BX>(g, fc, kappa, p, q, R, xcd_block(), gridDim.x);
}

// grid (nblocks, 3): one load case per block row
template <typename XT>
__global__ void __launch_bounds__(kBlock) k_fine_init_residual_case(Geom g, FineConsts fc,
                                                                    const float* __restrict__ kappa,
                                                                    const XT* __restrict__ x_,
                                                                    const float* __restrict__ xlo,
                                                                    float* __restrict__ rvec, Reduce R) {
  fine_init_residual_case_body<XT>(g, fc, kappa, x_, xlo, rvec, R, xcd_block(), gridDim.x, (int)blockIdx.y);
}

// the same by whole x-rows (fine_init_residual_rows_body), nx <= kBlock
template <typename XT>
__global__ void __launch_bounds__(kBlock) k_fine_init_residual_rows(Geom g, FineConsts fc,
                                                                    const float* __restrict__ kappa,
                                                                    const XT* __restrict__ x_,
                                                                    const float* __restrict__ xlo,
                                                                    float* __restrict__ rvec, Reduce R) {
  fine_init_residual_rows_body<XT>(g, fc, kappa, x_, xlo, rvec, R, xcd_block(), gridDim.x, (int)blockIdx.y);
}

__global__ void __launch_bounds__(kBlock) k_fine_kappa_h(Geom g, FineConsts fc, const float* __restrict__ kappa,
                                                         ChiRef chi, Reduce R, float* __restrict__ S6) {
  fine_kappa_h_body(g, fc, kappa, chi, R, xcd_block(), gridDim.x, S6);
}

__global__ void __launch_bounds__(kBlock) k_sens_from_energy(Geom g, const float* __restrict__ S6, float w0, float w1,
                                                             float w2, float w3, float w4, float w5,
                                                             float* __restrict__ sens, int pitch,
                                                             const float* __restrict__ scale) {
  const float w[6] = {w0, w1, w2, w3, w4, w5};
  sens_from_energy_body(g, S6, w, sens, pitch, stid(), scale);
}

__global__ void __launch_bounds__(kBlock) k_fine_sensitivity(Geom g, FineConsts fc, ChiRef chi,
                                                             float w0, float w1, float w2, float w3, float w4, float w5,
                                                             float* __restrict__ sens, int pitch,
                                                             const float* __restrict__ scale) {
  const float w[6] = {w0, w1, w2, w3, w4, w5};
  fine_sensitivity_body(g, fc, chi, w, sens, pitch, gtid(), scale);
}

__global__ void __launch_bounds__(kBlock) k_fine_energy6(Geom g, FineConsts fc, ChiRef chi,
                                                         float* __restrict__ S6) {
  fine_energy6_body(g, fc, chi, S6, gtid());
}

// The occupancy hint keeps the fully unrolled colour loop from holding
// every node's loads in flight at once (which costs occupancy); the 30 KB
// LDS footprint of a 32x4x8 brick allows five workgroups per CU.
// One tile and NR load cases per workgroup.
template <int BX, int BY, int BZ, int TR, int NR, bool RAG>
__global__ void __launch_bounds__(BX * TR) __attribute__((amdgpu_waves_per_eu(4, 8)))
k_fine_smooth_brick(Geom g, FineConsts fc, const float* __restrict__ kappa, const float* __restrict__ f,
                    const float* __restrict__ uin, float* __restrict__ uout, int sweeps, int forward, int zero_in,
                    int dot, Reduce RD) {
  constexpr int kParts = OTM_NRHS / NR;
  const int b = xcd_block(), k0 = (b % kParts) * NR;
  const size_t o = (size_t)k0 * (size_t)g.nn;
  fine_brick_body<BX, BY, BZ, TR, NR, RAG>(g, fc, kappa, f + o, uin + o, uout + o, sweeps, forward, zero_in, b / kParts,
                                           dot, RD, k0);
}

// A level whose edges are no multiples of a tile takes ragged tiles wherever
// their overhang wraps once (fine_ragged_x): faster at every size measured,
// from a solve of 12^3 (1192 -> 853 us) to 88 x 72 x 104 (3069 -> 2508).
// Exact colours remain for 8-wide cells, unequal sweep counts and the
// fallback.
//
// Up to this many tiles a launch takes one load case per workgroup: 8 tiles
// 10.3 -> 7.3 us. Three load cases against one, tiles of 256 threads: 128
// tiles 10.7 and 8.6 us, 192 10.8 and 10.4, 256 11.5 and 10.4, 384 12.8 and
// 14.0, 2048 28.6 and 44.7; of 128 threads: 216 tiles 11.9 and 11.6, 360 14.9
// and 14.0, 672 15.3 and 18.0. The curves cross between 256 and 384 tiles
// (360 and 672); the line lies below, where the gain is a fifth.
constexpr long long kFineOneMax = 128;

template <int BX, int BY, int BZ, int TR, bool RAG = false>
static void launch_fine_tile(hipStream_t s, const Geom& g, const FineConsts& fc, const float* kappa, const float* f,
                             const float* uin, float* uout, int sweeps, bool forward, bool zero_in, long long tiles,
                             const Reduce* dot) {
  const bool one = tiles <= kFineOneMax;
  const auto k = one ? k_fine_smooth_brick<BX, BY, BZ, TR, 1, RAG> : k_fine_smooth_brick<BX, BY, BZ, TR, OTM_NRHS, RAG>;
  hipLaunchKernelGGL(k, dim3((unsigned)(one ? OTM_NRHS * tiles : tiles)), dim3(BX * TR), 0, s, g, fc, kappa, f, uin,
                     uout, sweeps, forward ? 1 : 0, zero_in ? 1 : 0, dot ? 1 : 0, dot ? *dot : Reduce{});
}

void launch_fine_smooth_brick(hipStream_t s, const Geom& g, const FineConsts& fc, const float* kappa, const float* f,
                              const float* uin, float* uout, int sweeps, bool forward, bool zero_in, int v,
                              const Reduce* dot) {
  if (!fine_brick_ok(g, v)) throw std::invalid_argument("the cell does not tile with this fine tile shape");
  if (dot && !fine_brick_dot_ok(g, v)) throw std::invalid_argument("too many tiles for r.z in the smoother");
  const long long nt = fine_brick_tiles(g, v);
  if (v < 0) {
    const auto go = fine_ragged_x(g) == 32 ? launch_fine_tile<32, kFineBY, kFineBZ, kFineTR, true>
                                           : launch_fine_tile<16, kFineBY, kFineBZ, kFineTR, true>;
    go(s, g, fc, kappa, f, uin, uout, sweeps, forward, zero_in, nt, dot);
    return;
  }
  switch (v) {
    case 0: launch_fine_tile<32, 4, 8, 8>(s, g, fc, kappa, f, uin, uout, sweeps, forward, zero_in, nt, dot); break;
    case 1: launch_fine_tile<16, 4, 8, 8>(s, g, fc, kappa, f, uin, uout, sweeps, forward, zero_in, nt, dot); break;
    case 2: launch_fine_tile<32, 8, 4, 8>(s, g, fc, kappa, f, uin, uout, sweeps, forward, zero_in, nt, dot); break;
    case 3: launch_fine_tile<32, 4, 4, 4>(s, g, fc, kappa, f, uin, uout, sweeps, forward, zero_in, nt, dot); break;
    default: launch_fine_tile<32, 8, 8, 8>(s, g, fc, kappa, f, uin, uout, sweeps, forward, zero_in, nt, dot); break;
  }
}

void launch_fine_brick_dot_final(hipStream_t s, const Geom& g, const Reduce& R, int v) {
  launch_reduce_final(s, R, OTM_NRHS, (unsigned)fine_brick_tiles(g, v));
}

// ---- launchers ---------------------------------------------------------
static inline unsigned nblk(long long n) { return (unsigned)((n + kBlock - 1) / kBlock); }

void launch_fine_gs_color(hipStream_t s, const Geom& g, const FineConsts& fc, const float* kappa, const float* f,
                          float* u, int color) {
  const long long cnt = (long long)g.nx * (g.ny / 2) * (g.nz / 2);
  hipLaunchKernelGGL(k_fine_gs_color, dim3(nblk(cnt)), dim3(kBlock), 0, s, g, fc, kappa, f, u, color & 1, color >> 1);
}

void launch_fine_residual(hipStream_t s, const Geom& g, const FineConsts& fc, const float* kappa, const float* f,
                          const float* u, float* res) {
  const int bx = fine_tile_x(g);
  if (bx == 32)
    hipLaunchKernelGGL(k_fine_residual_tile<32>, dim3(fine_tiles(g, 32)), dim3(kBlock), 0, s, g, fc, kappa, f, u, res);
  else if (bx == 16)
    hipLaunchKernelGGL(k_fine_residual_tile<16>, dim3(fine_tiles(g, 16)), dim3(kBlock), 0, s, g, fc, kappa, f, u, res);
  else
    hipLaunchKernelGGL(k_fine_residual, dim3(nblk(g.nn)), dim3(kBlock), 0, s, g, fc, kappa, f, u, res);
}

// Levels that tile use the LDS-tiled kernel with its own workgroup count
// (fine_apply_tile_blocks); the reduction's partial count follows it.
void launch_fine_apply_dot(hipStream_t s, const Geom& g, const FineConsts& fc, const float* kappa, const float* p,
                           float* q, const Reduce& R, unsigned nblocks) {
  const int bx = fine_tile_x(g);
  if (bx) {
    const unsigned nb = fine_apply_tile_blocks(g, bx);
    if (bx == 32)
      hipLaunchKernelGGL(k_fine_apply_tile<32>, dim3(nb), dim3(kBlock), 0, s, g, fc, kappa, p, q, R);
    else
      hipLaunchKernelGGL(k_fine_apply_tile<16>, dim3(nb), dim3(kBlock), 0, s, g, fc, kappa, p, q, R);
    launch_reduce_final(s, R, OTM_NRHS, nb);
    return;
  }
  hipLaunchKernelGGL(k_fine_apply_dot, dim3(nblocks), dim3(kBlock), 0, s, g, fc, kappa, p, q, R);
  launch_reduce_final(s, R, OTM_NRHS, nblocks);
}

// The FP64 residual by whole x-rows where rows have at most kBlock nodes
// (3 new iterate values per node and case); longer rows take the pointwise
// form. An LDS-tiled form (180 VGPRs, two waves per SIMD) measured 25%
// slower than the pointwise one.
template <typename XT>
static void launch_init_residual_xt(hipStream_t s, const Geom& g, const FineConsts& fc, const float* kappa,
                                    const XT* x, const float* xlo, float* r, const Reduce& R, unsigned nblocks) {
  const dim3 grid(nblocks, OTM_NRHS), blk(kBlock);
  if (fine_rows_ok(g.nx))
    hipLaunchKernelGGL(k_fine_init_residual_rows<XT>, grid, blk, 0, s, g, fc, kappa, x, xlo, r, R);
  else
    hipLaunchKernelGGL(k_fine_init_residual_case<XT>, grid, blk, 0, s, g, fc, kappa, x, xlo, r, R);
  launch_reduce_final(s, R, 3 * OTM_NRHS, nblocks);
}

void launch_fine_init_residual(hipStream_t s, const Geom& g, const FineConsts& fc, const float* kappa,
                               const float* x, const float* xlo, float* r, const Reduce& R, unsigned nblocks) {
  launch_init_residual_xt<float>(s, g, fc, kappa, x, xlo, r, R, nblocks);
}

void launch_fine_init_residual(hipStream_t s, const Geom& g, const FineConsts& fc, const float* kappa,
                               const double* x, float* r, const Reduce& R, unsigned nblocks) {
  launch_init_residual_xt<double>(s, g, fc, kappa, x, nullptr, r, R, nblocks);
}

void launch_fine_kappa_h(hipStream_t s, const Geom& g, const FineConsts& fc, const float* kappa, const ChiRef& chi,
                         const Reduce& R, unsigned nblocks, float* S6) {
  hipLaunchKernelGGL(k_fine_kappa_h, dim3(nblocks), dim3(kBlock), 0, s, g, fc, kappa, chi, R, S6);
  launch_reduce_final(s, R, 6, nblocks);
}

void launch_sens_from_energy(hipStream_t s, const Geom& g, const float* S6, const float w[6], float* sens, int pitch,
                             const float* scale) {
  hipLaunchKernelGGL(k_sens_from_energy, dim3(nblk(g.nn)), dim3(kBlock), 0, s, g, S6, w[0], w[1], w[2], w[3], w[4],
                     w[5], sens, pitch, scale);
}

void launch_fine_sensitivity(hipStream_t s, const Geom& g, const FineConsts& fc, const ChiRef& chi, const float w[6],
                             float* sens, int pitch, const float* scale) {
  hipLaunchKernelGGL(k_fine_sensitivity, dim3(nblk(g.nn)), dim3(kBlock), 0, s, g, fc, chi, w[0], w[1], w[2], w[3],
                     w[4], w[5], sens, pitch, scale);
}

void launch_fine_energy6(hipStream_t s, const Geom& g, const FineConsts& fc, const ChiRef& chi, float* S6) {
  hipLaunchKernelGGL(k_fine_energy6, dim3(nblk(g.nn)), dim3(kBlock), 0, s, g, fc, chi, S6);
}

}  // namespace otm
