// Per-sample GMRES cycles on chip: interface between the adjoint driver and the
// kernels of gmres.hip.
#pragma once

#include "plan.hpp"

namespace purin {

constexpr int kGmrRestart = 32;  // restart lengths the cycle kernel takes (one lane per vector)
constexpr int kGmrGroup = 4;     // cycles enqueued between two host reads of the step counts

// One adjoint call's sample-major state.  A state vector of W = 2n + m elements
// holds y and ybar in the order of the sliced columns and d in the order of the
// sliced rows (purin_cp_plan::sl_cperm / sl_rperm); sample b's vectors start at
// b * Wp.
template <typename T>
struct Gmr {
  int n, m, W, restart;
  int64_t Wp;            // elements between vectors (a multiple of 16)
  // sliced rows and columns of the scaled kept matrix: slice s holds positions
  // 64 s .. 64 s + 63, entries off[s] .. off[s + 1) in [entry][lane] order, padded
  // with index n (rows) / m (columns), whose LDS element is zero
  int nsr, nsc;
  const int32_t* __restrict__ roff;
  const int32_t* __restrict__ coff;
  const uint16_t* __restrict__ ridx;
  const uint16_t* __restrict__ cidx;
  const T* __restrict__ rval;
  const T* __restrict__ cval;
  int64_t rstride, cstride;  // elements between samples' entries (0: shared)
  // operator scalars, or per element (DG): a, delta [n] and sigma [m] per sample
  T a, delta, sigma;
  const T* __restrict__ av;
  const T* __restrict__ dv;
  const T* __restrict__ sv;
  const T* __restrict__ mask;  // [n + m] per sample: clip derivative C, dual projection D
  const T* __restrict__ G;     // right-hand side
  T* X;                        // solution
  T* R;                        // residual
  T* Z;                        // raw basis, restart + 1 vectors per sample
  T* thr;                      // [batch] threshold
  T* rinf;                     // [batch] residual's largest entry
  T* xfin;                     // [batch] 1 where the solution is finite
  int32_t* total;              // [batch] Arnoldi steps over all cycles
  int32_t* ctrl;               // [kGmrGroup] steps of the group's cycles (largest over the batch)
};

// Whether the cycle kernel takes this plan and restart length.
bool gmr_fits(const purin_cp_plan* p, int64_t restart);

// One restart cycle for every unconverged sample: cycle ``c`` of a group whose
// earlier groups completed ``base`` steps of ``max_iterations``.
template <typename T>
int gmr_cycle(hipStream_t st, const Gmr<T>& A, int64_t batch, bool dg, int c, int64_t base,
              int64_t max_iterations);

}  // namespace purin
