// Same-size AMR blocks advanced together: the AMR branch of the reference's
// 2-D step (simulation/set_simulator.py:37-42, :107-111, and
// time_step/TVD_RK3.py:15-37), where flux_func, update_func and the
// chemistry are vmap-ed over a leading block axis.
//
// Layout: a batch of blocks is the reference's blk_data, (n_blk, 14, PX, PY)
// = U (12 planes) and aux (gamma, T) of each block, C-order; the stage
// entry's blocks carry their 3 ghost layers (PX = bnx + 6, PY = bny + 6,
// filled by the caller: jaxamr's get_ghost_block_data), the chemistry's do
// not (PX = bnx, PY = bny).  Each block has its own StepScalars: its LF
// maxima (vmap gives every block the nanmax over its own padded field) and
// health flags.  The temperature solves stop per cell.
#pragma once
#include <hip/hip_runtime.h>

#include "compact.hpp"
#include "stage.hpp"

namespace jh {

// Threads of a block stage kernel at most: tiles of up to 256 faces, sized to
// the AMR block (compact_tile).  Several small workgroups per CU cover one
// another's barriers: a whole FP64 step of 2500 blocks of 20 x 20 (a level in
// place) takes 694 us at 256 or 384 threads, 745 at 512, 799 at 192; the mixed
// step of 1000 blocks of 40 x 50 943 us at 256, 954 at 192, 1145 at 512.
constexpr int kBlkThreads = 256;
// Waves per SIMD its register budget allows.  FP32 takes 85 registers; held to 80 for
// the sixth wave it spills 3 of them (16 bytes a lane) and is the faster: the mixed
// level above 960 us with four or five, 939 with six.
template <typename Real> struct BlkWaves { static constexpr int value = 4; };
template <> struct BlkWaves<float> { static constexpr int value = 6; };

// LF maxima of stage `stage` of every block over its padded field
// (LF.py:10-11 under vmap): one workgroup per block, stored (not folded) into
// the block's StepScalars::amax[0][stage].
template <typename Real>
__global__ __launch_bounds__(256) void blocks_alpha_kernel(StepArgs<Real> a, int stage,
                                                           long long bs,
                                                           const Real* __restrict__ B) {
  __shared__ double red[8];
  const int b = blockIdx.x;
  const int P = (a.nx + 6) * (a.ny + 6);
  const Real* U = B + (size_t)b * bs;
  const Real* aux = U + (size_t)NU * P;
  const MechConst& c = *a.mc;
  double mx = 0.0, my = 0.0;
  for (int i = threadIdx.x; i < P; i += blockDim.x) {
    const Prim<double> q = cell_prim<double, true>(c, U + i, aux + i, P);
    mx = fmax(mx, nan_to_zero(fabs(q.u) + q.a));
    my = fmax(my, nan_to_zero(fabs(q.v) + q.a));
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    mx = fmax(mx, __shfl_xor(mx, off, 64));
    my = fmax(my, __shfl_xor(my, off, 64));
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) {
    red[wid] = mx;
    red[4 + wid] = my;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    double m = red[4 * threadIdx.x];
    for (int w = 1; w < 4; ++w) m = fmax(m, red[4 * threadIdx.x + w]);
    a.sc[b].amax[0][stage][threadIdx.x] = dbits(m);
  }
}

// One RK stage (MODE_RK) or the flux_func alone (MODE_RHS) of every block's
// interior: the compact stage body on a block's padded planes, the block's
// own maxima.  Jobs (block, tile) in XCD-contiguous order.  bs / bo: block
// strides of the inputs and of the output (12 planes per block for MODE_RHS).
// Bound by FP64 issue; the 64-column tile of the wide body leaves 44 of 64 lanes of
// a 20 x 20 block idle.
template <typename Real, int MODE>
__global__ __launch_bounds__(kBlkThreads) __attribute__((amdgpu_waves_per_eu(BlkWaves<Real>::value)))
void blocks_stage_kernel(StepArgs<Real> a, CompactTile ct, int stage, long long bs, long long bo,
                         const Real* Bs, const Real* Bn, Real* Bo) {
  extern __shared__ double dyn[];
  __shared__ MixTables mix;
  __shared__ double red[32];
  const int t = xcd_tile(blockIdx.x, gridDim.x), tiles = ct.tiles_x * ct.tiles_y;
  const int b = t / tiles, tile = t - b * tiles;
  const size_t P = (size_t)(a.nx + 6) * (a.ny + 6);
  StepArgs<Real> ab = a;
  ab.sc = a.sc + b;
  ab.parity = 0;
  const Real* Us = Bs + (size_t)b * bs;
  Real* Uo = Bo + (size_t)b * bo;
  compact_body<Real, MODE, 1, 1, ADDR_PAD>(ab, ct, stage, Us, Us + NU * P, Bn + (size_t)b * bs, Uo,
                                           Uo + NU * P, tile, blockDim.x,
                                           reinterpret_cast<Real*>(dyn), mix, red);
}

// The same by the wide stage body on kBlkRows x 64 tiles, bit for bit: for many blocks
// that fill its columns (blocks_wide).  Fewer halo cells a cell, and in FP32 runs of
// faces that share their differences: a mixed stage of 256 blocks of 64 x 64 takes 137
// us with it and 159 with compact tiles, an FP64 one 188 and 211.
constexpr int kBlkRows = 8;
template <typename Real, int MODE>
__global__ __launch_bounds__(Tile<kBlkRows>::NT) __attribute__((amdgpu_waves_per_eu(4)))
void blocks_stage_wide_kernel(StepArgs<Real> a, int stage, int tiles, long long bs, long long bo,
                              const Real* Bs, const Real* Bn, Real* Bo) {
  __shared__ StageLds<Real, kBlkRows> L;
  const int t = xcd_tile(blockIdx.x, gridDim.x);
  const int b = t / tiles, tile = t - b * tiles;
  const size_t P = (size_t)(a.nx + 6) * (a.ny + 6);
  StepArgs<Real> ab = a;
  ab.sc = a.sc + b;
  ab.parity = 0;
  const Real* Us = Bs + (size_t)b * bs;
  Real* Uo = Bo + (size_t)b * bo;
  stage_body<Real, MODE, kBlkRows, RECON_WENO5, SPLIT_LF, Real, false, false, true>(
      ab, stage, Us, Us + NU * P, Bn + (size_t)b * bs, Uo, Uo + NU * P, tile, L);
}

// One RK stage of a uniform level's blocks read in place: the halo of a block
// comes from the other blocks' interiors through the level's index table and
// the output is the interiors alone, so no padded copy is filled and no ghost
// ring is written (lv: tables and strides; Uo: (n_blk, 14, nx, ny)).
template <typename Real>
__global__ __launch_bounds__(kBlkThreads) __attribute__((amdgpu_waves_per_eu(BlkWaves<Real>::value)))
void level_stage_kernel(StepArgs<Real> a, CompactTile ct, int stage, LevelMap<Real> lv,
                        const Real* Us, const Real* Un, Real* Uo) {
  extern __shared__ double dyn[];
  __shared__ MixTables mix;
  __shared__ double red[32];
  const int t = xcd_tile(blockIdx.x, gridDim.x), tiles = ct.tiles_x * ct.tiles_y;
  const int b = t / tiles, tile = t - b * tiles;
  const size_t n = (size_t)a.nx * a.ny;
  StepArgs<Real> ab = a;
  ab.sc = a.sc + b;
  Real* Ub = Uo + (size_t)b * (NU + 2) * n;
  compact_body<Real, MODE_RK, 1, 1, ADDR_LEVEL>(ab, ct, stage, Us, nullptr, Un, Ub, Ub + NU * n,
                                                tile, blockDim.x, reinterpret_cast<Real*>(dyn),
                                                mix, red, &lv, b);
}

// |u| + a and |v| + a of every interior cell of a level (two planes of ncell)
// and each block's maxima of them into its stage-0 slots (the later stages'
// slots are cleared): what the level's stage kernels take the LF maxima from.
// One workgroup per block.
template <typename Real>
__global__ __launch_bounds__(256) void level_speeds_kernel(StepArgs<Real> a, long long sb,
                                                           long long splane, long long sr,
                                                           const Real* __restrict__ U,
                                                           double* __restrict__ spd, int ncell) {
  __shared__ double red[8];
  const int n = a.nx * a.ny, b = blockIdx.x;
  double mx = 0.0, my = 0.0;
  for (int l = threadIdx.x; l < n; l += blockDim.x) {
    const int x = l / a.ny, i = b * n + l;
    const Real* p = U + b * sb + x * sr + (l - x * a.ny);
    const Prim<double> q = cell_prim<double, true>(*a.mc, p, p + NU * splane, splane);
    const double sx = nan_to_zero(fabs(q.u) + q.a), sy = nan_to_zero(fabs(q.v) + q.a);
    spd[i] = sx;
    spd[ncell + i] = sy;
    mx = fmax(mx, sx);
    my = fmax(my, sy);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    mx = fmax(mx, __shfl_xor(mx, off, 64));
    my = fmax(my, __shfl_xor(my, off, 64));
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) {
    red[wid] = mx;
    red[4 + wid] = my;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    double m = red[4 * threadIdx.x];
    for (int w = 1; w < 4; ++w) m = fmax(m, red[4 * threadIdx.x + w]);
    a.sc[b].amax[0][0][threadIdx.x] = dbits(m);
    a.sc[b].amax[0][1][threadIdx.x] = 0ull;
    a.sc[b].amax[0][2][threadIdx.x] = 0ull;
  }
}

// The ghost layers of a stage's output blocks, as the reference computes
// them over the padded arrays (its rhs is zero there, TVD_RK3.py:21-35):
// U_out = the stage's combination of U_n and U_s, aux_out = update_aux from
// the stage input's T; MODE_RHS writes zeros (flux_func's jnp.pad).  Grid:
// (ring cells / 256, n_blk).
template <typename Real, int MODE>
__global__ __launch_bounds__(256) void blocks_ring_kernel(StepArgs<Real> a, int stage,
                                                          long long bs, long long bo,
                                                          const Real* __restrict__ Bs,
                                                          const Real* __restrict__ Bn,
                                                          Real* __restrict__ Bo) {
  __shared__ MixTables mix;
  const MechConst& c = *a.mc;
  if (MODE == MODE_RK) load_mix_tables(c, mix);
  __syncthreads();
  const int b = blockIdx.y;
  const int nx = a.nx, ny = a.ny, PY = ny + 6, P = (nx + 6) * PY;
  const int nring = P - nx * ny;
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned int fl = 0u;
  if (r < nring) {
    // rows 0-2 and nx+3..nx+5 whole, then the 6 ghost columns of rows 3..nx+2
    int px, py;
    if (r < 6 * PY) {
      const int row = r / PY;
      px = row < 3 ? row : nx + row;
      py = r - row * PY;
    } else {
      const int k = r - 6 * PY, row = k / 6, col = k - row * 6;
      px = 3 + row;
      py = col < 3 ? col : ny + col;
    }
    const int o = px * PY + py;
    Real* Uo = Bo + (size_t)b * bo;
    if (MODE == MODE_RHS) {
#pragma unroll
      for (int v = 0; v < NU; ++v) Uo[(size_t)v * P + o] = (Real)0;
    } else {
      const Real* Us = Bs + (size_t)b * bs;
      const Real* Un = Bn + (size_t)b * bs;
      double un[NU];
#pragma unroll
      for (int v = 0; v < NU; ++v) {
        const double us = (double)Us[(size_t)v * P + o];
        if (stage == 0) {
          un[v] = us + 0.0;
        } else {
          const double u0 = (double)Un[(size_t)v * P + o];
          if (stage == 1) un[v] = (3.0 / 4.0) * u0 + (1.0 / 4.0) * (us + 0.0);
          else un[v] = (1.0 / 3.0) * u0 + (2.0 / 3.0) * (us + 0.0);
        }
        Uo[(size_t)v * P + o] = (Real)un[v];
        un[v] = (double)(Real)un[v];
      }
      const double rho = un[0], ir = rcp(rho);
      const double u = un[1] * ir, v = un[2] * ir;
      const double e = un[3] * ir - 0.5 * (u * u + v * v);
      double Y[JH_NS];
#pragma unroll
      for (int k = 0; k < JH_NS - 1; ++k) Y[k] = un[4 + k] * ir;
      const double R = fill_Y_get_R(c, Y);
      double T = (double)Us[(size_t)(NU + 1) * P + o];
      double gamma;
      const bool conv = halley_T(mix, Y, R, e, T, gamma);
      Uo[(size_t)NU * P + o] = (Real)gamma;
      Uo[(size_t)(NU + 1) * P + o] = (Real)T;
      fl = halley_flags(rho, e, R, T, gamma, conv);
    }
  }
  raise_flags(a.sc + b, fl);
}

// Chemistry and final update_aux of every block's interior, in place
// (set_simulator.py:107-111): blocks (n_blk, 14, nx, ny).  Grid: all cells /
// 256 (a grid of whole workgroups per block left a fifth of the lanes idle at
// 400 cells a block).
template <typename Real>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void blocks_chem_kernel(StepArgs<Real> a, long long bs, Real* B, int n_blk) {
  __shared__ MixTables mix;
  __shared__ GibbsTables gt;
  chem_body<Real, CHEM_STEP, false, false, true>(a, B, B + (size_t)NU * a.nx * a.ny, nullptr,
                                                 nullptr, blockIdx.x, nullptr, nullptr, mix, gt, bs,
                                                 n_blk);
}

// Ghost refill of same-size blocks tiling one uniform level: out[b][v][p]
// (padded blocks, P = (bnx + 6)(bny + 6) cells each) = the interior cell
// idx[b P + p] of the level (flat index block * bnx * bny + x * bny + y) of
// plane v, times the cell's momentum sign (su for v = 1, sv for v = 2).
// The source is addressed by strides (block, plane, row; columns
// contiguous), so a padded stage output's interior view needs no copy.
// Grid: (ceil(n_blk P / 256), NV).
template <typename Real>
__global__ __launch_bounds__(256) void blocks_fill_kernel(
    const Real* __restrict__ src, long long sb, long long sv, long long sr, int bnx, int bny,
    const int* __restrict__ idx, const Real* __restrict__ su, const Real* __restrict__ svg,
    Real* __restrict__ out, int n_blk, int P) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int v = blockIdx.y;
  if (i >= (long long)n_blk * P) return;
  const long long b = i / P, p = i - b * P;
  const int col = idx[i], B = bnx * bny;
  const int cb = col / B, loc = col - cb * B, lx = loc / bny, ly = loc - lx * bny;
  Real x = src[cb * sb + v * sv + lx * sr + ly];
  if (v == 1) x *= su[i];
  else if (v == 2) x *= svg[i];
  out[(b * NV + v) * P + p] = x;
}

}  // namespace jh
