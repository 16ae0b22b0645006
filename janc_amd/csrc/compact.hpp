// Stage kernel for small pieces: small grids and AMR blocks.
//
// stage_kernel's tile is 64 columns wide (a wave per row) and walks the 12
// variables one after another behind two block barriers each: a grid of a few
// thousand cells fills a handful of CUs with one long serial block each, and
// a 20 x 20 AMR block leaves 44 of its 64 lanes idle.  Here a tile is R x C
// cells of any shape, its cells and faces dealt to the threads one each, and
// the variables are shared out to G groups of threads that work at the same
// time.  The arithmetic of a cell and of a face is stage_body's, so the states
// are its states bit for bit.
//
// What bounds it: on a small grid one block's chain (state loads, split
// fluxes, a face's WENO, the temperature solve), so the chain is made as short
// as the variables allow; on AMR levels FP64 / FP32 issue, so the tile is made
// to fill its waves (one cell, one x face and one y face per thread).  Whole
// steps, before and after: 128 x 32 FP64 155 -> 46 us, 256 x 64 mixed 122 -> 49
// us; a level of 2500 FP64 blocks of 20 x 20 2276 -> 659 us, of 1000 mixed
// blocks of 40 x 50 1608 -> 938 us.
#pragma once
#include <hip/hip_runtime.h>

#include "stage.hpp"

namespace jh {

// Where a tile's halo cells come from: ghost strips, the source cells of
// copy-kind sides, the ghost layers of a padded AMR block, or the interiors
// of the other blocks of a uniform level through its index table.
enum Addr : int { ADDR_STRIP = 0, ADDR_MIRROR = 1, ADDR_PAD = 2, ADDR_LEVEL = 3 };

// A uniform level of same-size blocks read in place (ADDR_LEVEL): entry
// b P + p of idx is the level's interior cell (flat block * nx * ny + x * ny +
// y) behind padded cell p of block b, su / sv its momentum signs; interior
// cells are at block * sb + x * sr + y of every plane (stride sv_), the
// cells' |u| + a and |v| + a in two planes of spd.
template <typename Real>
struct LevelMap {
  const int* __restrict__ idx;
  const Real* __restrict__ su;
  const Real* __restrict__ sv;
  const double* __restrict__ spd;   // speeds of the stage's input
  double* __restrict__ spd_out;     // speeds of its output (null: not wanted)
  long long sb, splane, sr;         // strides of the stage's input
  long long nb, nplane, nr;         // strides of the step's input (U^n)
  int ncell;                        // interior cells of the level
};

// Tile shape and the shared memory of one block, chosen on the host.
struct CompactTile {
  int R, C;                  // rows along x, columns along y
  int tiles_x, tiles_y;
  __host__ __device__ int hx() const { return (R + 6) * C; }
  __host__ __device__ int hy() const { return R * (C + 6); }
  __host__ __device__ int fx() const { return (R + 1) * C; }
  __host__ __device__ int fy() const { return R * (C + 1); }
  __host__ __device__ int cells() const { return R * C; }
  __host__ __device__ int halo() const { return 6 * (R + C); }
  // elements of one group's split fluxes and faces
  __host__ __device__ int group_len() const { return 2 * hx() + 2 * hy() + fx() + fy(); }
};

// Elements (of the state's type) of a block's dynamic shared memory: per
// group the split fluxes and faces; with several groups also the primitives
// of the region and the tile's new state.
template <int G>
__host__ __device__ inline int compact_lds(const CompactTile& t) {
  return G * t.group_len() + (G > 1 ? 4 * (t.cells() + t.halo()) + NU * t.cells() : 0);
}

template <typename Real, int MODE, int G, int NH, int ADDR>
__device__ __forceinline__ void compact_body(const StepArgs<Real>& a, const CompactTile& ct,
                                             int stage, const Real* __restrict__ Us,
                                             const Real* __restrict__ auxs, const Real* Un,
                                             Real* Uo, Real* __restrict__ auxo, int tile, int ntg,
                                             Real* lds, MixTables& mix, double* red,
                                             const LevelMap<Real>* lv = nullptr, int blk = 0) {
  using W = Real;
  const MechConst& c = *a.mc;
  if (MODE != MODE_RHS) load_mix_tables(c, mix);   // read after the phase barriers
  const int nx = a.nx, ny = a.ny;
  const int R = ct.R, C = ct.C;
  const int t = threadIdx.x;
  // group and thread of the group: groups are whole waves
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int g = G == 1 ? 0 : w / (ntg >> 6);
  const int tg = G == 1 ? t : t - g * ntg;
  if constexpr (ADDR == ADDR_MIRROR) {
    if (stage == 0 && tile == 0) zero_slots(a.sc, a.parity ^ 1);
  }
  const int x0 = (tile / ct.tiles_y) * R, y0 = (tile % ct.tiles_y) * C;
  const double dt = step_dt(a);
  constexpr double sc = LfScale<W>::value;   // split fluxes scaled as stage_body's
  constexpr W hs = (W)(0.5 * sc);
  const double idx = 1.0 / sc / a.dx, idy = 1.0 / sc / a.dy;
  // ---- the thread's cells: slot 0 = interior cell tg, then halo cells ----
  constexpr int NS = 1 + NH;
  const int ncell = ct.cells(), nhalo = ct.halo();
  const int xr = tg / C, yc = tg - xr * C;
  const auto halo_cell = [&](int h, int& lx, int& ly) {   // tile-relative, -3..
    if (h < 6 * C) {
      const int hr = h / C;
      lx = hr < 3 ? hr - 3 : R + hr - 3;
      ly = h - hr * C;
    } else {
      const int k = h - 6 * C, r = k / 6, pos = k - 6 * r;
      lx = r;
      ly = pos < 3 ? pos - 3 : C + pos - 3;
    }
  };
  const auto find = [&](int gx, int gy, unsigned int& f) -> CellRef<Real> {
    f = 0u;
    if constexpr (ADDR == ADDR_PAD) return locate_padded<Real>(a, Us, auxs, gx, gy);
    else if constexpr (ADDR == ADDR_MIRROR) return locate_src<Real>(a, Us, auxs, gx, gy, f);
    else if constexpr (ADDR == ADDR_STRIP) return locate<Real>(a, Us, auxs, gx, gy);
    else {
      CellRef<Real> r;
      r.stride = 0;                    // planes are lv->splane apart (plane)
      const bool inx = gx >= 0 && gx < nx, iny = gy >= 0 && gy < ny;
      r.ok = gx >= -3 && gx < nx + 3 && gy >= -3 && gy < ny + 3;
      long long o = 0;
      if (r.ok && inx && iny) {
        o = (long long)blk * lv->sb + gx * lv->sr + gy;
      } else if (r.ok) {
        const int i = blk * (nx + 6) * (ny + 6) + (gx + 3) * (ny + 6) + gy + 3;
        const int s = lv->idx[i], B = nx * ny, cb = s / B, l = s - cb * B, lx = l / ny;
        o = cb * lv->sb + lx * lv->sr + (l - lx * ny);
        f = (lv->su[i] < (Real)0 ? 1u : 0u) | (lv->sv[i] < (Real)0 ? 2u : 0u);
      }
      r.u = Us + o;
      r.x = r.u + NU * lv->splane;
      return r;
    }
  };
  // Element v planes from a cell.  The planes of a level's interiors are the
  // caller's view: their stride may be of any size.
  const auto plane = [&](const CellRef<Real>& r, int v) -> Real {
    if constexpr (ADDR == ADDR_LEVEL) return r.u[v * lv->splane];
    else return r.u[(size_t)v * r.stride];
  };
  CellRef<Real> ref[NS];
  Prim<W> q[NS];
  Real nxt[NS];
  bool has[NS], xhalo[NS];
  int li[NS];                 // LDS index: x region (slot 0 and x halo) or y region
  unsigned int flips = 0u;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    int lx, ly;
    if (s == 0) {
      has[0] = tg < ncell;
      lx = xr;
      ly = yc;
      xhalo[0] = true;
      li[0] = tg + 3 * C;
    } else {
      const int h = tg + (s - 1) * ntg;
      has[s] = h < nhalo;
      halo_cell(h, lx, ly);
      xhalo[s] = h < 6 * C;
      li[s] = xhalo[s] ? (lx + 3) * C + ly : lx * (C + 6) + ly + 3;
    }
    unsigned int f = 0u;
    // a tile's last rows or columns may lie past the grid: no cell there
    ref[s] = find(x0 + lx, y0 + ly, f);
    if (!has[s]) ref[s].ok = false;
    flips |= f << (2 * s);
  }
  if constexpr (G == 1) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (!ref[s].ok) continue;
      if constexpr (ADDR == ADDR_LEVEL)
        q[s] = cell_prim<W, false>(c, ref[s].u, ref[s].x, lv->splane);
      else
        q[s] = cell_prim<W, false>(c, ref[s].u, ref[s].x, ref[s].stride);
    }
  } else {
    // the region's primitives once per block, through LDS
    W* sP = lds + G * ct.group_len();
    const int nreg = ncell + nhalo;
    for (int i = t; i < nreg; i += blockDim.x) {
      int lx, ly;
      if (i < ncell) {
        lx = i / C;
        ly = i - lx * C;
      } else {
        halo_cell(i - ncell, lx, ly);
      }
      unsigned int f;
      const CellRef<Real> r = find(x0 + lx, y0 + ly, f);
      if (r.ok) {
        const Prim<W> p = cell_prim<W, false>(c, r.u, r.x, r.stride);
        sP[i] = p.rho;
        sP[nreg + i] = p.u;
        sP[2 * nreg + i] = p.v;
        sP[3 * nreg + i] = p.p;
      }
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int i = s == 0 ? tg : ncell + tg + (s - 1) * ntg;
      if (ref[s].ok) {
        q[s].rho = sP[i];
        q[s].u = sP[nreg + i];
        q[s].v = sP[2 * nreg + i];
        q[s].p = sP[3 * nreg + i];
      }
    }
  }
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    if (!ref[s].ok) continue;
    if ((flips >> (2 * s)) & 1u) q[s].u = -q[s].u;
    if ((flips >> (2 * s)) & 2u) q[s].v = -q[s].v;
  }
  double alx, aly;
  if constexpr (ADDR == ADDR_LEVEL) {
    // the block's LF maxima: its interior cells' (reduced by the producer) and
    // its ghost cells', which are copies of interior cells with the momenta
    // negated at most, through the index table; after the state's reads, which
    // cover the table's (mixed level of 1000 blocks: 958 -> 945 us a step)
    const int PY = ny + 6, P = (nx + 6) * PY, ring = P - nx * ny;
    double mx = 0.0, my = 0.0;
    for (int r = t; r < ring; r += blockDim.x) {
      int p;
      if (r < 6 * PY) {                    // rows 0-2 and nx+3..nx+5 whole
        p = r < 3 * PY ? r : r + nx * PY;
      } else {                             // the 6 ghost columns of the rows between
        const int k = r - 6 * PY, row = k / 6, col = k - row * 6;
        p = (3 + row) * PY + (col < 3 ? col : ny + col);
      }
      const int s = lv->idx[(size_t)blk * P + p];
      mx = fmax(mx, lv->spd[s]);
      my = fmax(my, lv->spd[lv->ncell + s]);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      mx = fmax(mx, __shfl_xor(mx, off, 64));
      my = fmax(my, __shfl_xor(my, off, 64));
    }
    const int nw = blockDim.x >> 6;
    if ((t & 63) == 0) {
      red[w] = mx;
      red[16 + w] = my;
    }
    __syncthreads();
    alx = fmax(bitsd(a.sc->amax[0][stage][0]), red[0]);
    aly = fmax(bitsd(a.sc->amax[0][stage][1]), red[16]);
    for (int i = 1; i < nw; ++i) {
      alx = fmax(alx, red[i]);
      aly = fmax(aly, red[16 + i]);
    }
  } else {
    alx = bitsd(a.sc->amax[a.parity][stage][0]);
    aly = bitsd(a.sc->amax[a.parity][stage][1]);
  }
  const W hax = hs * (W)(Real)alx, hay = hs * (W)(Real)aly;

  const int gx = x0 + xr, gy = y0 + yc;
  const bool own = has[0] && gx < nx && gy < ny;
  const int n = ADDR == ADDR_PAD ? (nx + 6) * (ny + 6) : nx * ny;
  const int oidx = ADDR == ADDR_PAD ? (gx + 3) * (ny + 6) + gy + 3 : gx * ny + gy;
  // U^n of the thread's cell
  const long long unidx = ADDR == ADDR_LEVEL ? (long long)blk * lv->nb + gx * lv->nr + gy : oidx;
  const long long unstride = ADDR == ADDR_LEVEL ? lv->nplane : n;

  W* sHxp = lds + g * ct.group_len();
  W* sHxm = sHxp + ct.hx();
  W* sHyp = sHxm + ct.hx();
  W* sHym = sHyp + ct.hy();
  W* sFx = sHym + ct.hy();
  W* sFy = sFx + ct.fx();
  W* sU = lds + G * ct.group_len() + 4 * (ncell + nhalo);
  const int hyi = xr * (C + 6) + yc + 3;             // own cell in the y region
  const bool xface = tg < ct.fx(), yface = tg < ct.fy();
  const int fr = tg / (C + 1), ybase = fr * (C + 6) + tg - fr * (C + 1);
  const int fyi = xr * (C + 1) + yc;                 // own cell's low y face

  // phase 1 of variable cv: split fluxes into LDS (CLS = min(cv, 4))
  const auto split = [&](auto K, const W (&uc)[NS]) {
    constexpr int CLS = decltype(K)::value;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (!has[s]) continue;
      W ucv = uc[s];
      if constexpr (CLS == 1 || CLS == 2) {
        if ((flips >> (2 * s + CLS - 1)) & 1u) ucv = -ucv;
      }
      if (s == 0 || xhalo[s]) {
        W hp = (W)0, hm = (W)0;
        if (ref[s].ok) {
          const W hF = hs * phys_flux<W>(CLS, 0, q[s], ucv);
          hp = fma(hax, ucv, hF);
          hm = fma(-hax, ucv, hF);
        }
        sHxp[li[s]] = hp;
        sHxm[li[s]] = hm;
      }
      if (s == 0 || !xhalo[s]) {
        W hp = (W)0, hm = (W)0;
        if (ref[s].ok) {
          const W hG = hs * phys_flux<W>(CLS, 1, q[s], ucv);
          hp = fma(hay, ucv, hG);
          hm = fma(-hay, ucv, hG);
        }
        const int yi = s == 0 ? hyi : li[s];
        sHyp[yi] = hp;
        sHym[yi] = hm;
      }
    }
  };
  constexpr int NVG = NU / G;                        // variables of a group
  static_assert(NU % G == 0, "groups share the variables evenly");
  const int cv0 = g * NVG;
#pragma unroll
  for (int s = 0; s < NS; ++s)
    nxt[s] = ref[s].ok ? plane(ref[s], cv0) : (Real)0;
#pragma unroll 1
  for (int k = 0; k < NVG; ++k) {
    const int cv = cv0 + k;
    W uc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) uc[s] = (W)nxt[s];
    switch (cv) {            // wave-uniform
      case 0: split(std::integral_constant<int, 0>{}, uc); break;
      case 1: split(std::integral_constant<int, 1>{}, uc); break;
      case 2: split(std::integral_constant<int, 2>{}, uc); break;
      case 3: split(std::integral_constant<int, 3>{}, uc); break;
      default: split(std::integral_constant<int, 4>{}, uc);
    }
    __syncthreads();
    if (k + 1 < NVG) {
#pragma unroll
      for (int s = 0; s < NS; ++s)
        if (ref[s].ok) nxt[s] = plane(ref[s], cv + 1);
    }
    W u0n = (W)0;
    if (MODE != MODE_RHS && stage != 0 && own) u0n = (W)Un[unidx + cv * unstride];
    // ---- phase 2: one x face and one y face per thread ----
    if (xface) {
      const W* p = sHxp + tg;
      const W* m = sHxm + tg;
      sFx[tg] = weno5_lf(p[0], p[C], p[2 * C], p[3 * C], p[4 * C], m[C], m[2 * C], m[3 * C],
                         m[4 * C], m[5 * C]);
    }
    if (yface) {
      const W* p = sHyp + ybase;
      const W* m = sHym + ybase;
      sFy[tg] = weno5_lf(p[0], p[1], p[2], p[3], p[4], m[1], m[2], m[3], m[4], m[5]);
    }
    __syncthreads();
    // ---- phase 3: divergence + RK combine, as stage_body ----
    if (own) {
      const double dF = (double)sFx[tg + C] - (double)sFx[tg];
      const double dG = (double)sFy[fyi + 1] - (double)sFy[fyi];
      const double rhs = dt * (-(dF * idx + dG * idy));
      double un;
      if (MODE == MODE_RHS) {
        un = rhs;
      } else if (stage == 0) {
        un = (double)uc[0] + rhs;
      } else {
        const double u0 = (double)u0n, ucd = (double)uc[0];
        if (stage == 1) un = (3.0 / 4.0) * u0 + (1.0 / 4.0) * (ucd + rhs);
        else un = (1.0 / 3.0) * u0 + (2.0 / 3.0) * (ucd + rhs);
      }
      Uo[(size_t)cv * n + oidx] = (Real)un;
      if constexpr (G > 1 && MODE != MODE_RHS) sU[cv * ncell + tg] = (Real)un;
    }
  }
  if (MODE == MODE_RHS) return;

  // ---- update_aux and the next stage's LF maxima, one cell per thread ----
  if constexpr (G > 1) __syncthreads();
  double mx = 0.0, my = 0.0;
  unsigned int fl = 0u;
  if (own && g == 0) {
    const Real* un = G > 1 ? sU + tg : Uo + oidx;
    const int st = G > 1 ? ncell : n;
    const double rho = (double)un[0], ir = rcp(rho);
    const double u = (double)un[st] * ir, v = (double)un[2 * st] * ir;
    const double e = (double)un[3 * st] * ir - 0.5 * (u * u + v * v);
    double Y[JH_NS];
#pragma unroll
    for (int k = 0; k < JH_NS - 1; ++k) Y[k] = (double)un[(4 + k) * st] * ir;
    const double Rg = fill_Y_get_R(c, Y);
    double T = (double)(ADDR == ADDR_LEVEL ? plane(ref[0], NU + 1) : ref[0].x[ref[0].stride]);
    double gamma;
    const bool conv = halley_T(mix, Y, Rg, e, T, gamma);
    auxo[oidx] = (Real)gamma;
    auxo[n + oidx] = (Real)T;
    fl = halley_flags(rho, e, Rg, T, gamma, conv);
    const double gs = (double)(Real)gamma, Ts = (double)(Real)T;
    const double p = rho * Rg * Ts;
    const double snd = sqrt(gs * p * ir);
    mx = nan_to_zero(fabs(u) + snd);
    my = nan_to_zero(fabs(v) + snd);
    if constexpr (ADDR == ADDR_LEVEL) {
      if (lv->spd_out) {
        lv->spd_out[blk * nx * ny + oidx] = mx;
        lv->spd_out[lv->ncell + blk * nx * ny + oidx] = my;
      }
    }
  }
  raise_flags(a.sc, fl);
  if constexpr (ADDR != ADDR_PAD) {
    if (stage < 2) {
      if constexpr (ADDR == ADDR_LEVEL) __syncthreads();   // red was read at the start
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        mx = fmax(mx, __shfl_xor(mx, off, 64));
        my = fmax(my, __shfl_xor(my, off, 64));
      }
      const int nw = ntg >> 6;          // waves of group 0, which hold the maxima
      if ((t & 63) == 0 && g == 0) {
        red[w] = mx;
        red[16 + w] = my;
      }
      __syncthreads();
      if (t < 2) {
        double m = red[16 * t];
        for (int i = 1; i < nw; ++i) m = fmax(m, red[16 * t + i]);
        const unsigned long long mb = dbits(m);
        unsigned long long* dst = &a.sc->amax[a.parity][stage + 1][t];
        if (mb > __hip_atomic_load(dst, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
          atomicMax(dst, mb);
      }
    }
  }
}

// Tile of at most ntg cells, x faces and y faces (one of each per thread) and
// nh * ntg halo cells that covers nx x ny in the fewest tiles; of equals the
// one with the smallest region.
inline CompactTile compact_tile(int nx, int ny, int ntg, int nh) {
  CompactTile best{0, 0, 0, 0};
  long long bt = 0, br = 0;
  for (int C = 1; C <= ny && C < ntg; ++C) {
    int R = ntg / C - 1;                                  // (R + 1) C <= ntg
    if (R > ntg / (C + 1)) R = ntg / (C + 1);             // R (C + 1) <= ntg
    if (R > nh * ntg / 6 - C) R = nh * ntg / 6 - C;       // 6 (R + C) <= nh ntg
    if (R > nx) R = nx;
    if (R < 1) continue;
    const int tx = (nx + R - 1) / R, ty = (ny + C - 1) / C;
    R = (nx + tx - 1) / tx;                               // even rows
    if ((ny + ty - 1) / ty != C) continue;                // an even split comes by itself
    const long long tiles = (long long)tx * ty, reg = (long long)R * C + 6 * (R + C);
    if (!best.R || tiles < bt || (tiles == bt && reg < br)) {
      best = CompactTile{R, C, tx, ty};
      bt = tiles;
      br = reg;
    }
  }
  return best;
}

// LDS: dynamic, compact_lds<G>(ct) elements of Real.
template <typename Real, int MODE, int G, int NH, int NT, int ADDR>
__global__ __launch_bounds__(NT) void compact_stage_kernel(
    StepArgs<Real> a, CompactTile ct, int ntg, int stage, const Real* __restrict__ Us,
    const Real* __restrict__ auxs, const Real* Un, Real* Uo, Real* __restrict__ auxo) {
  extern __shared__ double dyn[];
  __shared__ MixTables mix;
  __shared__ double red[32];
  compact_body<Real, MODE, G, NH, ADDR>(a, ct, stage, Us, auxs, Un, Uo, auxo,
                                        xcd_tile(blockIdx.x, gridDim.x), ntg,
                                        reinterpret_cast<Real*>(dyn), mix, red);
}

}  // namespace jh
