// Batched launch of many independent cases (uneven grid sizes) of the step.
//
// Each case keeps its own state, stage buffers, ghost strips and reduction
// scalars; a device array of CaseDesc describes them.  One launch per
// kernel kind covers every case: a block finds its case by binary search in a
// prefix-sum table of per-case block counts, loads that case's arguments and runs the same
// per-tile / per-cell body as the single-case kernels, so every case's result
// is bit-identical to advancing it alone.
#pragma once
#include <hip/hip_runtime.h>

#include "stage.hpp"

namespace jh {

template <typename Real>
struct CaseDesc {
  StepArgs<Real> a;          // geometry, BCs, strips, scalars of the case
  Real* U;                   // state (12 planes), advanced in place
  Real* aux;                 // (gamma, T)
  Real* U1;                  // RK stage buffers
  Real* U2;
  Real* A1;
  Real* A2;
};

// Case owning flat block index b: off[k] <= b < off[k+1] (off has ncase+1
// entries, off[0] = 0).  b is wave-uniform, so this runs on the scalar unit.
__device__ __forceinline__ int find_case(const int* __restrict__ off, int ncase, int b) {
  int lo = 0, hi = ncase;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= b) lo = mid;
    else hi = mid;
  }
  return lo;
}

// A pointer read from a case's descriptor, known to be device memory.  A
// pointer that comes from memory is otherwise a generic one: its loads go
// through the flat path, which waits on the LDS counter too, and uniform ones
// are not scalar loads.
template <typename T>
__device__ __forceinline__ T* device_ptr(T* p) {
  using Global = __attribute__((address_space(1))) T;
  return (T*)(Global*)(unsigned long long)p;
}

// A case's arguments.  The mechanism is the kernel's own argument, the same for
// every case, so its constants are scalar loads as in the single-case kernels.
// 64 mixed cases of 7.0M cells in all: chemistry 1029 -> 859 us (700 since), stage
// kernel 939 -> 661 us a launch.
template <typename Real>
__device__ __forceinline__ StepArgs<Real> case_args(const CaseDesc<Real>& d,
                                                    const MechConst* __restrict__ mc, int parity,
                                                    double dt_fixed, double cfl) {
  StepArgs<Real> a = d.a;
  a.mc = mc;
  a.sc = device_ptr(d.a.sc);
#pragma unroll
  for (int s = 0; s < 4; ++s) a.g[s] = device_ptr(d.a.g[s]);
  a.parity = parity;
  a.dt_fixed = dt_fixed;
  a.cfl = cfl;
  return a;
}

// Zero the parity's reduction slots of every case (thread k -> case k).
template <typename Real>
__global__ void reset_batch_kernel(const CaseDesc<Real>* __restrict__ d, int ncase, int parity) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= ncase) return;
  StepScalars* sc = d[k].a.sc;
#pragma unroll
  for (int i = 0; i < 6; ++i) (&sc->amax[parity][0][0])[i] = 0ull;
  sc->cmax[parity] = 0ull;
}

template <typename Real>
__global__ __launch_bounds__(256) void reduce_batch_kernel(
    const CaseDesc<Real>* __restrict__ d, const int* __restrict__ off,
    const MechConst* __restrict__ mc, int ncase, int parity, double dt_fixed, double cfl) {
  __shared__ double red[4];
  __shared__ unsigned long long redb[4];
  const int k = find_case(off, ncase, blockIdx.x);
  const StepArgs<Real> a = case_args(d[k], mc, parity, dt_fixed, cfl);
  reduce_body<Real>(a, device_ptr(d[k].U), device_ptr(d[k].aux), parity, 1,
                    blockIdx.x - off[k], off[k + 1] - off[k], red, redb);
}

template <typename Real>
__global__ __launch_bounds__(kBcThreads) void bc_batch_kernel(
    const CaseDesc<Real>* __restrict__ d, const int* __restrict__ off,
    const MechConst* __restrict__ mc, int ncase, int stage, int parity, double dt_fixed,
    double cfl) {
  __shared__ double red[4];
  const int k = find_case(off, ncase, blockIdx.x);
  const CaseDesc<Real>& cd = d[k];
  const StepArgs<Real> a = case_args(cd, mc, parity, dt_fixed, cfl);
  const Real* U = stage == 0 ? cd.U : stage == 1 ? cd.U1 : cd.U2;
  const Real* A = stage == 0 ? cd.aux : stage == 1 ? cd.A1 : cd.A2;
  bc_body<Real>(a, device_ptr(U), device_ptr(A), stage, blockIdx.x - off[k], red);
}

// Stage kernel over the flat tile list of all cases, one block per tile.  Tile
// numbers go through xcd_tile, so each XCD walks a contiguous run of the list:
// whole cases or long runs of one case's x-adjacent tiles.  (A persistent grid
// that loops over the list, sized to the resident blocks, takes 940 us a launch
// where this takes 661: it holds every case argument and the loop's state
// across the tile body and spills.)
// MIRROR: every case's sides are copy kinds and the halo is read from the
// source cells (no ghost-strip launches).
template <typename Real, int TX, int WPE, bool MIRROR = false>
__global__ __launch_bounds__(Tile<TX>::NT) __attribute__((amdgpu_waves_per_eu(WPE)))
void stage_batch_kernel(const CaseDesc<Real>* __restrict__ d, const int* __restrict__ off,
                        const MechConst* __restrict__ mc, int ncase, int stage, int parity,
                        double dt_fixed, double cfl) {
  __shared__ StageLds<Real, TX> L;
  const int t = xcd_tile(blockIdx.x, gridDim.x);
  const int k = find_case(off, ncase, t);
  const CaseDesc<Real>& cd = d[k];
  const StepArgs<Real> a = case_args(cd, mc, parity, dt_fixed, cfl);
  const Real* Us = stage == 0 ? cd.U : stage == 1 ? cd.U1 : cd.U2;
  const Real* As = stage == 0 ? cd.aux : stage == 1 ? cd.A1 : cd.A2;
  Real* Uo = stage == 0 ? cd.U1 : stage == 1 ? cd.U2 : cd.U;
  Real* Ao = stage == 0 ? cd.A1 : stage == 1 ? cd.A2 : cd.aux;
  stage_body<Real, MODE_RK, TX, RECON_WENO5, SPLIT_LF, Real, false, MIRROR>(
      a, stage, device_ptr(Us), device_ptr(As), device_ptr(cd.U), device_ptr(Uo), device_ptr(Ao),
      t - off[k], L);
}

// Chemistry + final update_aux for every case; dt_hist (optional) is
// (ncase, hist_len) row-major, step s written at column s.
template <typename Real>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void chem_batch_kernel(const CaseDesc<Real>* __restrict__ d, const int* __restrict__ off,
                       const MechConst* __restrict__ mc, int ncase, int parity, double dt_fixed,
                       double cfl, double* dt_hist, int hist_len, int s) {
  __shared__ unsigned long long red[12];
  const int k = find_case(off, ncase, blockIdx.x);
  const CaseDesc<Real>& cd = d[k];
  const StepArgs<Real> a = case_args(cd, mc, parity, dt_fixed, cfl);
  __shared__ MixTables mix;
  __shared__ GibbsTables gt;
  chem_body<Real, CHEM_STEP>(a, device_ptr(cd.U), device_ptr(cd.aux), nullptr,
                             dt_hist ? dt_hist + (size_t)k * hist_len + s : nullptr,
                             blockIdx.x - off[k], red, nullptr, mix, gt);
}

}  // namespace jh
