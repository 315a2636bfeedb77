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
  int rparts, cparts;    // wavefronts that share a slice's entries (1: short rows / columns)
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

// Whether a workgroup's LDS holds the products' vectors (n + m up to 16,130 in fp64, 36,600 in
// fp32).
bool gmr_holds(const purin_cp_plan* p);
// The largest batch that runs one workgroup per sample (0: none), for GMRES of this restart
// length or the dense layer's BiCGSTAB.
int64_t gmr_batch(const purin_cp_plan* p, int64_t restart, bool dense);

// One restart cycle for every unconverged sample: cycle ``c`` of a group whose
// earlier groups completed ``base`` steps of ``max_iterations``.
template <typename T>
int gmr_cycle(hipStream_t st, const Gmr<T>& A, int64_t batch, bool dg, int c, int64_t base,
              int64_t max_iterations);

// BiCGSTAB over the whole batch as one vector (fixed_point.py:8-40), one workgroup per
// sample: the vectors rhat, p, q, s, t in the basis slots 0..4, the scalars in ``sc``
// (kBiScalars), per-sample partial sums in ``part`` [3][batch], a ticket counter.
enum BiScalar { kBiBS = 0, kBiAtol2, kBiRho, kBiAlpha, kBiOmega, kBiRhoN, kBiAlphaN, kBiOmegaN,
                kBiBeta, kBiSS, kBiK, kBiIt, kBiGo, kBiScalars };
template <typename T>
struct GmrBi {
  T* sc;
  T* part;
  int32_t* ticket;
  int64_t batch;
  T tol, atol;
  int64_t max_iterations;
};
constexpr int kBiGroup = 16;  // iterations enqueued between two host reads

template <typename T>
int gmr_bicgstab(hipStream_t st, const Gmr<T>& A, const GmrBi<T>& B, int iterations, bool start);

// The wavefronts that share a slice in the kernels' products (for Gmr::rparts, cparts).
int gmr_parts(int64_t W, int slices, int widest);

}  // namespace purin
