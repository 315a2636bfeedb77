// The CP loop with one workgroup per sample: interface between the forward driver
// and the kernels of solo.hip.
#pragma once

#include "plan.hpp"

namespace purin {

// Which steps and objective the loop uses.
enum SoloMode {
  kSoloShared = 0,  // the plan's scalar schedule, q = 1, c = -yhat
  kSoloValues = 1,  // per-sample steps, q = 1, c = -yhat
  kSoloQP = 2,      // per-sample steps, general q and c
};

// Per-sample arrays are batch-minor (element e of sample b at e * Bp + b), as the
// streaming passes read them: each is loaded once, at launch.
template <typename T>
struct Solo {
  int n, m, me;
  int64_t Bp, batch, iters;
  // sliced rows and columns (purin_cp_plan::sl_*)
  int nsr, nsc;
  const int32_t* __restrict__ roff;
  const int32_t* __restrict__ coff;
  const int32_t* __restrict__ rperm;
  const int32_t* __restrict__ cperm;
  const uint16_t* __restrict__ ridx;
  const uint16_t* __restrict__ cidx;
  const T* __restrict__ rval;  // slice order, shared by the samples; or nullptr:
  const T* __restrict__ cval;
  const T* __restrict__ RV;    // kept CSR / CSC entries, [entry * vbp + b * (vbp > 1)]
  const T* __restrict__ CV;    // through the slices' source maps
  const int32_t* __restrict__ rsrc;
  const int32_t* __restrict__ csrc;
  int64_t vbp;
  const T* __restrict__ tgt;   // yhat, or c (QP)
  const T* __restrict__ Q;     // q (QP)
  const T* __restrict__ R;     // scaled right-hand sides
  const T* __restrict__ LO;
  const T* __restrict__ HI;
  int shared_bounds;           // one copy of the bounds, [n]
  const T* __restrict__ sched; // [iters][4] = sigma, a, delta, theta (kSoloShared)
  const T* __restrict__ step0; // [5][Bp] = tau, sigma, a, delta, theta of iteration 0
  const T* __restrict__ gam;   // [Bp] gamma of the accelerated update, or nullptr (1)
  int accel;
  T tol;                       // or per sample from tolv [Bp]
  const T* __restrict__ tolv;
  int32_t* done;
  int32_t* count;
  T* Y;                        // n x Bp; QP: holds y0
  T* D;                        // m x Bp; holds the initial duals
};

// Whether the kernel takes this plan, and pays for this batch.  values: the coefficients
// are per sample.
bool solo_fits(const purin_cp_plan* p, int64_t batch, bool early, bool values);

template <typename T>
int solo_launch(hipStream_t st, const purin_cp_plan* p, const Solo<T>& A, int mode, bool early);

// The projection's loop for problems whose vectors fill a CU's LDS (Solo's fields; the
// thread walks several rows and columns).  Targets, right-hand sides and bounds are
// sample-major in slice order: each is read every iteration.
template <typename T>
struct SoloWide {
  int n, m, me;
  int64_t Bp, batch, iters;
  int nsr, nsc;
  const int32_t* __restrict__ roff;
  const int32_t* __restrict__ coff;
  const int32_t* __restrict__ rperm;
  const int32_t* __restrict__ cperm;
  const uint16_t* __restrict__ ridx;
  const uint16_t* __restrict__ cidx;
  const T* __restrict__ rval;
  const T* __restrict__ cval;
  const T* __restrict__ TG;   // [batch][n]
  const T* __restrict__ RR;   // [batch][m]
  const T* __restrict__ LO;   // [n], or [batch][n] (bstride n)
  const T* __restrict__ HI;
  int64_t bstride;
  const T* __restrict__ sched;
  T tol;
  const T* __restrict__ tolv;
  int32_t* done;
  int32_t* count;
  T* Y;
  T* D;
};
// Whether a workgroup's LDS holds the plan's vectors, whether the kernel takes it, and whether
// it pays for this batch.
bool solo_wide_holds(const purin_cp_plan* p);
bool solo_wide_can(const purin_cp_plan* p, bool early);
bool solo_wide_fits(const purin_cp_plan* p, int64_t batch, bool early);
template <typename T>
int solo_wide_launch(hipStream_t st, const purin_cp_plan* p, const SoloWide<T>& A, bool early);

// The dense adapter's loop (factored prox, no freezing, no stationarity test): every sample
// iterates until the last is accepted.  A row is shared by 2^lr lanes, a column by 2^lc.
template <typename T>
struct SoloDense {
  int n, m, me, lr, lc, rw, cw;  // rw / cw: entries of a lane's row / column (at most kSoloDenseW)
  int64_t Bp, batch, iters;
  const int32_t* __restrict__ rptr;
  const int32_t* __restrict__ ridx;
  const int32_t* __restrict__ cptr;
  const int32_t* __restrict__ cidx;
  const T* __restrict__ RV;  // kept CSR / CSC entries, [entry * vbp + b * (vbp > 1)]
  const T* __restrict__ CV;
  int64_t vbp;
  const T* __restrict__ Q;
  const T* __restrict__ C;
  const T* __restrict__ R;
  const T* __restrict__ LO;
  const T* __restrict__ HI;
  const T* __restrict__ step0;  // [5][Bp]
  const T* __restrict__ gam;    // [Bp] or nullptr
  int accel;
  const T* __restrict__ tolv;
  T* Y;                         // n x Bp: y0, then y
  T* YB;                        // n x Bp: ybar between the two launches
  T* D;
  int32_t* done;
  int32_t* count;
  int32_t* last;                // the iteration at which the last sample is accepted
};
bool solo_dense_fits(const purin_cp_plan* p);
template <typename T>
int solo_dense_launch(hipStream_t st, const purin_cp_plan* p, SoloDense<T> A, bool early);

}  // namespace purin
