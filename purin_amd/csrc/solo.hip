// CP loop for small problems and batches: one workgroup per sample, one thread per
// row and per column, the thread's matrix entries in registers.
//
// The tile kernels of resident.hpp stream the shared matrix from L2 every iteration
// through 16 wavefronts whatever the problem's size, so below a few hundred
// thousand entries of work an iteration is latency: L2 loads, three barriers of 16
// wavefronts and a decision phase, 2.3-2.9 us.  Here
//   * the workgroup has as many wavefronts as the problem's rows or columns fill,
//     so small batches use more of the chip and small problems wait for less;
//   * a thread's first W entries of its row and of its column are in registers,
//     the rest (the widest slices only) in LDS, so an iteration touches no memory
//     beyond LDS: gather, sum, update, two barriers;
//   * the stop test trails the loop: a wavefront of its own sums and judges iteration
//     k's terms while the others run iteration k + 1, so the test is not on the path of
//     the iterates.  The state of two iterations back is kept, and a sample accepted at
//     k returns exactly that state and count.  (With all 16 wavefronts taken by rows or
//     columns, or with four or eight where one more would cost a workgroup per CU
//     (solo_block), each reduces its own terms and the last one judges.)
// One iteration (kernels.py:91-150): the column pass gathers d+, forms y+ and its
// diagnostics; the row pass gathers y+: K y+, the residual, and the next d+ from
// K ybar = (1 + theta) K y+ - theta K y (resident.hpp, k_resident_early).  Without the
// stop test the passes are k_resident's.
#include <algorithm>
#include <type_traits>

#include "solo.hpp"

#include "resident.hpp"

namespace purin {

namespace {

constexpr int kSoloMax = 1024;  // rows / columns: one thread each
constexpr int kSoloW = 8;       // matrix entries of a row and of a column in registers

// sum over N register entries: coefficient times the LDS element at its byte offset
template <int N, typename T, int W>
__device__ __forceinline__ T dot_regs(const T (&v)[W], const uint32_t (&ix)[W / 2],
                                      const unsigned char* lds) {
  T x[N], acc = T(0);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const uint32_t off = (k & 1) ? ix[k / 2] >> 16 : ix[k / 2] & 0xffffu;
    x[k] = *reinterpret_cast<const T*>(lds + off);
  }
#pragma unroll
  for (int k = 0; k < N; ++k) acc = __builtin_elementwise_fma(v[k], x[k], acc);
  return acc;
}

// A slice's sum: groups of 4 entries in registers (the count is the wavefront's),
// then the entries past W from LDS.  FOUR: four of those in flight.  Most kernels' loops the
// compiler unrolls by itself, by eight; the fp64 ones with the stop test that are short of
// registers it leaves at one entry, 140 cycles each (us per iteration of the QP, a row of 200
// entries, B = 256: 12.0, with FOUR 5.6; the others with FOUR 3.8 -> 5.1).
template <bool FOUR, typename T, int W>
__device__ __forceinline__ T slice_sum(const T (&v)[W], const uint32_t (&ix)[W / 2], int groups,
                                       const unsigned char* lds, const T* rv, const uint16_t* ri,
                                       int rest) {
  T acc = groups <= 1 ? dot_regs<4>(v, ix, lds) : dot_regs<8>(v, ix, lds);
  int k = 0;
  if constexpr (FOUR) {
    for (; k + 4 <= rest; k += 4) {
      T c[4], x[4];
      uint32_t at[4];
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        at[h] = ri[(k + h) * 64];
        c[h] = rv[(k + h) * 64];
      }
#pragma unroll
      for (int h = 0; h < 4; ++h) x[h] = *reinterpret_cast<const T*>(lds + at[h]);
#pragma unroll
      for (int h = 0; h < 4; ++h) acc = __builtin_elementwise_fma(c[h], x[h], acc);
    }
  }
  for (; k < rest; ++k)
    acc = __builtin_elementwise_fma(rv[k * 64], *reinterpret_cast<const T*>(lds + ri[k * 64]), acc);
  return acc;
}

// [a's sum over the wavefront in lanes 0-31, b's in lanes 32-63]
template <typename T>
__device__ __forceinline__ T two_sums(T a, T b) {
  constexpr int N = sizeof(T) / 4;
  typedef uint32_t U __attribute__((ext_vector_type(N)));
  U x = __builtin_bit_cast(U, a), y = __builtin_bit_cast(U, b);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const auto r = __builtin_amdgcn_permlane32_swap(x[i], y[i], false, false);
    x[i] = r[0];
    y[i] = r[1];
  }
  T v = __builtin_bit_cast(T, x) + __builtin_bit_cast(T, y);
  x = y = __builtin_bit_cast(U, v);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const auto r = __builtin_amdgcn_permlane16_swap(x[i], y[i], false, false);
    x[i] = r[0];
    y[i] = r[1];
  }
  v = __builtin_bit_cast(T, x) + __builtin_bit_cast(T, y);
  return row16_combine(v, OpAdd());
}

template <typename T>
__device__ __forceinline__ T wave_fmax(T a) {
  constexpr int N = sizeof(T) / 4;
  typedef uint32_t U __attribute__((ext_vector_type(N)));
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    U x = __builtin_bit_cast(U, a), y = x;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const auto r = h == 0 ? __builtin_amdgcn_permlane32_swap(x[i], y[i], false, false)
                            : __builtin_amdgcn_permlane16_swap(x[i], y[i], false, false);
      x[i] = r[0];
      y[i] = r[1];
    }
    a = __builtin_fmax(__builtin_bit_cast(T, x), __builtin_bit_cast(T, y));
  }
  return row16_combine(a, OpFMax());
}

// Entries past the first W of every slice, in LDS.
__host__ __device__ inline int rest_of(int width, int W) { return width > W ? width - W : 0; }

// The wavefronts' partial terms of a lane, in order.  The loads of up to 8 wavefronts are in
// flight together: one after the other they held up the iterations of all (us per iteration
// with the stop test, fp64: n = 300 1.06 -> 0.81, n = 400 1.05 -> 0.75, n = 777 1.35 -> 1.10,
// n = 950 1.31 -> 1.02; fp32 n = 777 1.16 -> 0.92).  Eight wavefronts or fewer go four at a
// time: with all at once the burst delays the others' gathers (n = 500 0.95 -> 1.03).
template <int N, typename T>
__device__ __forceinline__ void add_some(const T* pt, int NT, T& pri, T& dual, T& mx) {
  T a[N], b[N], c[N];
#pragma unroll
  for (int w = 0; w < N; ++w) {
    a[w] = pt[w * 64];
    b[w] = pt[NT + w * 64];
    c[w] = pt[2 * NT + w * 64];
  }
#pragma unroll
  for (int w = 0; w < N; ++w) {
    pri += a[w];
    dual += b[w];
    mx = __builtin_fmax(mx, c[w]);
  }
}
template <typename T>
__device__ __forceinline__ void add_parts(const T* pt, int NW, int NT, T& pri, T& dual, T& mx) {
  if (NW > 8) {
    add_some<8>(pt, NT, pri, dual, mx);
    pt += 8 * 64;
  }
  for (int w = (NW > 8 ? NW - 8 : NW) >> 2; w > 0; --w) {
    add_some<4>(pt, NT, pri, dual, mx);
    pt += 4 * 64;
  }
  if (NW & 2) {
    add_some<2>(pt, NT, pri, dual, mx);
    pt += 2 * 64;
  }
  if (NW & 1) add_some<1>(pt, NT, pri, dual, mx);
}

// Up to 1024 threads, so up to 128 VGPRs.
// HELP: the workgroup has one wavefront more than its rows or columns fill, for the stop test.
template <typename T, int W, int MODE, bool EARLY, bool HELP>
__global__ __launch_bounds__(1024) void k_solo(Solo<T> A) {
  extern __shared__ __align__(16) unsigned char lds[];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int NW = (blockDim.x >> 6) - (HELP ? 1 : 0);  // wavefronts of rows and columns
  const int NT = NW * 64;
  const int64_t b = blockIdx.x, Bp = A.Bp;
  const int n = A.n, m = A.m;
  const int j = t < n ? A.cperm[t] : -1, i = t < m ? A.rperm[t] : -1;
  if (b >= A.batch) {  // padding samples: zero state (the whole workgroup)
    if (j >= 0) A.Y[(int64_t)j * Bp + b] = T(0);
    if (i >= 0) A.D[(int64_t)i * Bp + b] = T(0);
    return;
  }
  constexpr bool QP = MODE == kSoloQP, PS = MODE != kSoloShared;
  constexpr bool FOUR = sizeof(T) == 8 && EARLY && (PS || !HELP);
  const T zero = T(0), half = T(0.5), inf = T(__builtin_inf());
  // LDS: Gy [n] | zero | Gd [m] | zero | partials [16][4] or (HELP) [2][3][NT] | verdict |
  // rest values | rest offsets
  T* Gy = reinterpret_cast<T*>(lds);
  T* Gd = Gy + n + 1;
  T* red = Gd + m + 1;
  T* fl = red + (HELP ? 6 * NT : 64);
  volatile int* flag = reinterpret_cast<volatile int*>(fl);
  T* restv = fl + 2;
  int nrest = 0, rbase = 0, cbase = 0;
  for (int s = 0; s < A.nsr; ++s) {
    if (s == wave) rbase = nrest;
    nrest += rest_of((A.roff[s + 1] - A.roff[s]) >> 6, W) * 64;
  }
  for (int s = 0; s < A.nsc; ++s) {
    if (s == wave) cbase = nrest;
    nrest += rest_of((A.coff[s + 1] - A.coff[s]) >> 6, W) * 64;
  }
  uint16_t* resti = reinterpret_cast<uint16_t*>(restv + nrest);
  // this wavefront's slices
  const bool has_r = wave < A.nsr, has_c = wave < A.nsc;
  const int ro = has_r ? A.roff[wave] : 0, co = has_c ? A.coff[wave] : 0;
  const int rw = has_r ? (A.roff[wave + 1] - ro) >> 6 : 0, cw = has_c ? (A.coff[wave + 1] - co) >> 6 : 0;
  const int rgr = (rw < W ? rw + 3 : W) >> 2, cgr = (cw < W ? cw + 3 : W) >> 2;
  const int rrest = rest_of(rw, W), crest = rest_of(cw, W);
  T rv[W], cv[W];
  uint32_t rx[W / 2], cx[W / 2];
  const uint32_t zr = (uint32_t)n * sizeof(T), zc = (uint32_t)(n + 1 + m) * sizeof(T);
  const uint32_t base_d = (uint32_t)(n + 1) * sizeof(T);
  auto value = [&](const T* shared, const T* own, const int32_t* src, int e) -> T {
    if (shared) return shared[e];
    const int k = src[e];
    return k < 0 ? T(0) : own[(int64_t)k * A.vbp + (A.vbp > 1 ? b : 0)];
  };
#pragma unroll
  for (int k = 0; k < W; ++k) {
    const int er = ro + k * 64 + lane, ec = co + k * 64 + lane;
    const bool okr = k < rw, okc = k < cw;
    rv[k] = okr ? value(A.rval, A.RV, A.rsrc, er) : zero;
    cv[k] = okc ? value(A.cval, A.CV, A.csrc, ec) : zero;
    const uint32_t xr = okr ? (uint32_t)A.ridx[er] * (uint32_t)sizeof(T) : zr;
    const uint32_t xc = okc ? base_d + (uint32_t)A.cidx[ec] * (uint32_t)sizeof(T) : zc;
    if (k & 1) {
      rx[k / 2] |= xr << 16;
      cx[k / 2] |= xc << 16;
    } else {
      rx[k / 2] = xr;
      cx[k / 2] = xc;
    }
  }
  for (int k = 0; k < rrest; ++k) {
    const int e = ro + (W + k) * 64 + lane;
    restv[rbase + k * 64 + lane] = value(A.rval, A.RV, A.rsrc, e);
    resti[rbase + k * 64 + lane] = (uint16_t)(A.ridx[e] * sizeof(T));
  }
  for (int k = 0; k < crest; ++k) {
    const int e = co + (W + k) * 64 + lane;
    restv[cbase + k * 64 + lane] = value(A.cval, A.CV, A.csrc, e);
    resti[cbase + k * 64 + lane] = (uint16_t)(base_d + A.cidx[e] * sizeof(T));
  }
  const T* rrv = restv + rbase + lane;
  const T* crv = restv + cbase + lane;
  const uint16_t* rri = resti + rbase + lane;
  const uint16_t* cri = resti + cbase + lane;
  // the thread's column and row
  const T tg = j >= 0 ? A.tgt[(int64_t)j * Bp + b] : zero;
  const T lo = j >= 0 ? A.LO[A.shared_bounds ? j : (int64_t)j * Bp + b] : zero;
  const T hi = j >= 0 ? A.HI[A.shared_bounds ? j : (int64_t)j * Bp + b] : zero;
  const T q = QP ? (j >= 0 ? A.Q[(int64_t)j * Bp + b] : T(1)) : T(1);
  const bool odd = lo != lo || hi != hi || lo > hi;  // a NaN or crossed bound
  T y = QP ? (j >= 0 ? A.Y[(int64_t)j * Bp + b] : zero) : tg;  // y0 = ybar0
  const T rr = i >= 0 ? A.R[(int64_t)i * Bp + b] : zero;
  T d = i >= 0 ? A.D[(int64_t)i * Bp + b] : zero;
  const bool ineq = i >= A.me;
  // per-sample steps, the same in every thread
  T tau = zero, sig = zero, th = T(1), gam = T(1), pa = zero, pd = zero;
  if constexpr (PS) {
    tau = res_uniform(A.step0[b]);
    sig = res_uniform(A.step0[Bp + b]);
    pa = res_uniform(A.step0[2 * Bp + b]);
    pd = res_uniform(A.step0[3 * Bp + b]);
    th = res_uniform(A.accel ? A.step0[4 * Bp + b] : T(1));
    gam = res_uniform(A.gam ? A.gam[b] : T(1));
  }
  auto prox = [&]() {  // the general-q prox a, delta (kernels.py:68-73)
    if constexpr (QP) {
      pa = EARLY ? T(1) / (T(1) + tau * q) : res_recip(T(1) + tau * q);
      pd = tau * pa;
    }
  };
  auto advance = [&]() {  // the accelerated update (kernels.py:279-283)
    if constexpr (PS) {
      if (A.accel) {
        T g1[1] = {gam}, t1[1] = {tau}, s1[1] = {sig}, h1[1] = {th}, a1[1], d1[1];
        res_qp_schedule<T, 1>(g1, t1, s1, h1, a1, d1);
        tau = t1[0];
        sig = s1[0];
        th = h1[0];
        if constexpr (!QP) {
          pa = a1[0];
          pd = d1[0];
        }
        prox();
      }
    }
  };
  prox();
  if (t < n) Gy[t] = y;
  if (t < m) Gd[t] = d;
  if (t == 0) {
    Gy[n] = zero;
    Gd[m] = zero;
    *flag = 0;
  }
  __syncthreads();
  typedef const __attribute__((address_space(4))) T* CP;
  const CP sched = (CP)A.sched;

  // s = a y - delta K^T d + delta yhat (or - delta c)
  auto primal_step = [&](T tt, T a, T delta) -> T {
    if constexpr (QP) {
      const T o = -delta * tg;
      return a * y - delta * tt + o;
    } else {
      return a * y - delta * tt + delta * tg;
    }
  };

  if constexpr (!EARLY) {
    // each iteration's scalars are loaded before the barrier that ends the previous one:
    // a scalar load outstanding among the gathers would make their waits wait for it too
    T f_sig = zero, f_a = zero, f_d = zero, f_th = zero;
    auto load = [&](int64_t k) {
      if constexpr (!PS) {
        f_sig = sched[4 * k];
        f_a = sched[4 * k + 1];
        f_d = sched[4 * k + 2];
        f_th = sched[4 * k + 3];
        asm volatile("" : "+s"(f_sig), "+s"(f_a), "+s"(f_d), "+s"(f_th));
      }
    };
    load(0);
    for (int64_t it = 0; it < A.iters; ++it) {
      const T sigma = PS ? sig : f_sig, a = PS ? pa : f_a, delta = PS ? pd : f_d,
              theta = PS ? th : f_th;
      if (has_r) {
        const T acc = slice_sum<FOUR, T, W>(rv, rx, rgr, lds, rrv, rri, rrest);
        T p = d + sigma * (acc - rr);
        if (ineq) p = res_pos(p);
        d = p;
        if (t < m) Gd[t] = p;
      }
      __syncthreads();
      if (has_c) {
        const T tt = slice_sum<FOUR, T, W>(cv, cx, cgr, lds, crv, cri, crest);
        const T s = primal_step(tt, a, delta);
        const T yn = odd ? clipp(s, lo, hi) : res_clip(s, lo, hi);
        if (t < n) Gy[t] = yn + theta * (yn - y);
        y = yn;
      }
      advance();
      if (it + 1 < A.iters) load(it + 1);
      __syncthreads();
    }
    if (j >= 0) A.Y[(int64_t)j * Bp + b] = y;
    if (i >= 0) A.D[(int64_t)i * Bp + b] = d;
    return;
  }

  // K y0 and the first d+
  T ky = zero;
  if (has_r) {
    ky = slice_sum<FOUR, T, W>(rv, rx, rgr, lds, rrv, rri, rrest);
    T p = d + (PS ? sig : sched[0]) * (ky - rr);
    if (ineq) p = res_pos(p);
    d = p;
    if (t < m) Gd[t] = p;
  }
  __syncthreads();
  const T tol = A.tolv ? A.tolv[b] : A.tol;
  const T one = T(1);
  auto judge = [&](T pri, T dual, T mx) -> bool {  // kernels.py:167-175, 260-278
    const T gap = maxp(pri - dual, zero) / maxp(one, maxp(absv(pri), absv(dual)));
    return finite(gap) && mx <= tol && gap <= tol;
  };
  if (HELP && wave == NW) {
    for (int64_t it = 0;; ++it) {
      if ((it >= 2 && __builtin_amdgcn_readfirstlane(*flag)) || it > A.iters) return;
      T pri = zero, dual = zero, mx = inf;
      if (it > 0) {
        const T* pt = red + ((it - 1) & 1) * 3 * NT + lane;
        mx = zero;
        add_parts(pt, NW, NT, pri, dual, mx);
      }
      __syncthreads();
      const T s2 = two_sums(pri, dual);
      const bool ok = judge(read_lane(s2, 0), read_lane(s2, 32), wave_fmax(mx));
      if (lane == 0) *flag = ok ? 1 : 0;
      __syncthreads();
    }
  }
  // the scalars of this iteration and the next sigma, loaded as in the loop above
  T f_a = zero, f_d = zero, f_th = zero, f_sn = zero;
  auto load = [&](int64_t k) {
    if constexpr (!PS) {
      const int64_t c = k < A.iters ? k : A.iters - 1, s = k + 1 < A.iters ? k + 1 : A.iters - 1;
      f_a = sched[4 * c + 1];
      f_d = sched[4 * c + 2];
      f_th = sched[4 * c + 3];
      f_sn = sched[4 * s];
      asm volatile("" : "+s"(f_a), "+s"(f_d), "+s"(f_th), "+s"(f_sn));
    }
  };
  load(0);
  T yp = y, dk = d, dkp = d;           // y and d+ one iteration back, d+ two back
  T q_pri = zero, q_dual = zero, q_max = inf;  // the last iteration's partials
  int64_t it = 0;
  bool accepted = false;
  for (;; ++it) {
    if (it >= 2 && __builtin_amdgcn_readfirstlane(*flag)) {  // the verdict on iteration it - 2
      accepted = true;
      break;
    }
    if (it > A.iters) break;  // one pass beyond the last judges the last
    const bool run = it < A.iters;
    const T r_pri = q_pri, r_dual = q_dual, r_max = q_max;
    yp = y;
    // ---- column pass, and the previous iteration's partials over the wavefront
    q_pri = q_dual = q_max = zero;
    if (run && has_c) {
      const T a = PS ? pa : f_a, delta = PS ? pd : f_d;
      const T tt = slice_sum<FOUR, T, W>(cv, cx, cgr, lds, crv, cri, crest);
      const T s = primal_step(tt, a, delta);
      const T yn = odd ? clipp(s, lo, hi) : res_clip(s, lo, hi);
      y = yn;
      if (t < n) {
        Gy[t] = yn;
        if constexpr (QP) {  // general q, c (kernels.py:158-174, 272-274)
          q_pri = half * q * yn * yn + tg * yn;
          const T tf = tg + tt;
          const T mz = q > T(1e-12) ? clipp(-tf / q, lo, hi) : (tf >= zero ? lo : hi);
          q_dual = half * q * (mz * mz) + tf * mz;
          T g = maxp(absv(yn - clipp(yn - ((q * yn + tg) + tt), lo, hi)),
                     maxp(maxp(lo - yn, zero), maxp(yn - hi, zero)));
          if (!finite(g)) g = inf;
          q_max = g;
        } else if (!odd) {  // q = 1, c = -yhat; see k_resident_early
          const T cq = -tg;
          q_pri = half * yn * yn + cq * yn;
          const T tf = cq + tt;
          const T mz = __builtin_fmin(__builtin_fmax(-tf, lo), hi);
          q_dual = half * mz * mz + tf * mz;
          q_max = __builtin_fmax(zero, absv(yn - mz));
        } else {
          const T cq = -tg;
          q_pri = half * yn * yn + cq * yn;
          const T tf = cq + tt;
          const T mz = clipp(-tf, lo, hi);
          q_dual = half * mz * mz + tf * mz;
          const T xs = yn - ((yn + cq) + tt);
          T g = maxp(absv(yn - clipp(xs, lo, hi)),
                     maxp(maxp(lo - yn, zero), maxp(yn - hi, zero)));
          if (!finite(g)) g = inf;
          q_max = g;
        }
      }
    }
    if constexpr (!HELP) {
      const T s2 = two_sums(r_pri, r_dual);
      const T mx = wave_fmax(r_max);
      if ((lane & 31) == 0) red[wave * 4 + (lane >> 5)] = s2;
      if (lane == 0) red[wave * 4 + 2] = mx;
    }
    __syncthreads();
    // ---- row pass, and the last wavefront's verdict on iteration it - 1
    dkp = dk;
    dk = d;
    const bool more = it + 1 < A.iters;
    const T theta = PS ? th : f_th;  // this iteration's; the steps then advance to the next
    if (PS && run) advance();
    if (run && has_r) {
      const T sigma_n = PS ? sig : f_sn;
      const T acc = slice_sum<FOUR, T, W>(rv, rx, rgr, lds, rrv, rri, rrest);
      if (t < m) {  // kernels.py:158-166; d * 0 is NaN for a non-finite d
        const T e = acc - rr, w = ineq ? zero : T(-1);
        q_max = __builtin_fmax(q_max, __builtin_fmax(e, w * e));
        q_dual = (q_dual - rr * d) - d * zero;
      }
      if (more) {
        T p = d + sigma_n * (((T(1) + theta) * acc - theta * ky) - rr);
        if (ineq) p = res_pos(p);
        d = p;
        if (t < m) Gd[t] = p;
      }
      ky = acc;
    }
    if constexpr (HELP) {
      T* pt = red + (it & 1) * 3 * NT + t;
      pt[0] = q_pri;
      pt[NT] = q_dual;
      pt[2 * NT] = q_max;
    } else if (wave == NW - 1) {
      const T* rl = red + (lane & 15) * 4;
      const bool in = (lane & 15) < NW;
      const T xp = row16_combine(in ? rl[0] : zero, OpAdd());
      const T xd = row16_combine(in ? rl[1] : zero, OpAdd());
      const T mx = row16_combine(in ? rl[2] : zero, OpFMax());
      const bool ok = it > 0 && judge(xp, xd, mx);
      if (lane == 0) *flag = ok ? 1 : 0;
    }
    load(it + 1);
    __syncthreads();
  }
  // accepted at iteration it - 2: its y and d+ are the ones of one iteration back
  if (accepted) {
    y = yp;
    dk = dkp;
  }
  if (j >= 0) A.Y[(int64_t)j * Bp + b] = y;
  if (i >= 0) A.D[(int64_t)i * Bp + b] = dk;
  if (t == 0) {
    A.count[b] = (int32_t)(accepted ? it - 1 : A.iters);
    A.done[b] = accepted ? 1 : 0;
  }
}

// ---------------------------------------------------------------------------
// Several rows and columns per thread: y, d and two copies of K y in LDS, the matrix, the
// targets, right-hand sides and bounds streamed from L2 (coalesced, in slice order).  The
// streaming passes it stands in for pad a batch to 128 (fp64) or 256 (fp32) samples and
// take four to six launches an iteration, and their time does not fall with the batch.
// What bounds it is the latency of those streams, so a wavefront keeps the loads of
// four slices in flight.
// ---------------------------------------------------------------------------
constexpr int kWideU = 4;  // slices of a wavefront in flight
constexpr int kWideThreads = 1024;

// sums of slices s0, s0 + 16, ... (kWideU of them): acc[u] = entries times x
template <typename T>
__device__ __forceinline__ void wide_sums(int s0, int ns, const int32_t* __restrict__ off,
                                          const uint16_t* __restrict__ idx,
                                          const T* __restrict__ val, const T* x,
                                          T (&acc)[kWideU]) {
  const int lane = threadIdx.x & 63;
  int o[kWideU], w[kWideU];
#pragma unroll
  for (int u = 0; u < kWideU; ++u) {
    const int s = s0 + 16 * u;
    o[u] = s < ns ? off[s] : 0;
    w[u] = s < ns ? (off[s + 1] - o[u]) >> 6 : 0;
    acc[u] = T(0);
  }
  // slices are in decreasing width, so the first is the widest of the four
  for (int k = 0; k < w[0]; k += 4) {
    T v[kWideU][4];
    int e[kWideU][4];
#pragma unroll
    for (int u = 0; u < kWideU; ++u) {
      if (k >= w[u]) continue;
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const int at = o[u] + (k + h < w[u] ? k + h : w[u] - 1) * 64 + lane;
        v[u][h] = val[at];
        e[u][h] = idx[at];
      }
    }
#pragma unroll
    for (int u = 0; u < kWideU; ++u) {
      if (k >= w[u]) continue;
#pragma unroll
      for (int h = 0; h < 4; ++h)
        if (k + h < w[u]) acc[u] = __builtin_elementwise_fma(v[u][h], x[e[u][h]], acc[u]);
    }
  }
}

template <typename T, bool EARLY>
__global__ __launch_bounds__(1024) void k_solo_wide(SoloWide<T> A) {
  extern __shared__ __align__(16) unsigned char lds[];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t b = blockIdx.x, Bp = A.Bp;
  const int n = A.n, m = A.m;
  if (b >= A.batch) {
    for (int e = t; e < n; e += 1024) A.Y[(int64_t)e * Bp + b] = T(0);
    for (int e = t; e < m; e += 1024) A.D[(int64_t)e * Bp + b] = T(0);
    return;
  }
  const T zero = T(0), one = T(1), half = T(0.5), inf = T(__builtin_inf());
  T* Gy = reinterpret_cast<T*>(lds);  // y [n] | zero
  T* Gd = Gy + n + 1;                 // d+ [m] | zero
  T* KY = Gd + m + 1;                 // K y of the previous y [m]
  // K y+ waits for the stop test's verdict in registers where a wavefront has one group of
  // row slices (m <= 4096), else in LDS
  const bool one_group = A.nsr <= 16 * kWideU;
  T* KN = KY + m;
  T* red = KN + (EARLY && !one_group ? m : 0);  // [16][4]
  const T* TG = A.TG + (size_t)b * n;
  const T* RR = A.RR + (size_t)b * m;
  const T* LO = A.LO + (size_t)b * A.bstride;
  const T* HI = A.HI + (size_t)b * A.bstride;
  for (int e = t; e < n; e += 1024) Gy[e] = TG[e];  // y0 = ybar0 = yhat
  for (int e = t; e < m; e += 1024) Gd[e] = A.D[(int64_t)A.rperm[e] * Bp + b];
  if (t == 0) Gy[n] = Gd[m] = zero;
  __syncthreads();
  typedef const __attribute__((address_space(4))) T* CP;
  const CP sched = (CP)A.sched;
  // K y0 and the first d+
  {
    const T sigma = sched[0];
    for (int s0 = wave; s0 < A.nsr; s0 += 16 * kWideU) {
      T acc[kWideU];
      wide_sums(s0, A.nsr, A.roff, A.ridx, A.rval, Gy, acc);
#pragma unroll
      for (int u = 0; u < kWideU; ++u) {
        const int i = (s0 + 16 * u) * 64 + lane;
        if (s0 + 16 * u >= A.nsr || i >= m) continue;
        T p = Gd[i] + sigma * (acc[u] - RR[i]);
        if (A.rperm[i] >= A.me) p = res_pos(p);
        Gd[i] = p;
        KY[i] = acc[u];
      }
    }
  }
  __syncthreads();
  const T tol = EARLY ? (A.tolv ? A.tolv[b] : A.tol) : zero;
  bool accepted = false;
  int64_t it = 0;
  for (; it < A.iters; ++it) {
    const T a = sched[4 * it + 1], delta = sched[4 * it + 2], theta = sched[4 * it + 3];
    const bool more = it + 1 < A.iters;
    const T sigma_n = more ? sched[4 * (it + 1)] : zero;
    T pri = zero, dual = zero, mx = zero;
    // ---- column pass: y+ and its diagnostics
    for (int s0 = wave; s0 < A.nsc; s0 += 16 * kWideU) {
      T tg[kWideU], lo[kWideU], hi[kWideU], acc[kWideU];
#pragma unroll
      for (int u = 0; u < kWideU; ++u) {
        const int j = (s0 + 16 * u) * 64 + lane;
        const bool in = s0 + 16 * u < A.nsc && j < n;
        tg[u] = in ? TG[j] : zero;
        lo[u] = in ? LO[j] : zero;
        hi[u] = in ? HI[j] : zero;
      }
      wide_sums(s0, A.nsc, A.coff, A.cidx, A.cval, Gd, acc);
#pragma unroll
      for (int u = 0; u < kWideU; ++u) {
        const int j = (s0 + 16 * u) * 64 + lane;
        if (s0 + 16 * u >= A.nsc || j >= n) continue;
        const T tt = acc[u];
        const bool odd = lo[u] != lo[u] || hi[u] != hi[u] || lo[u] > hi[u];
        const T s = a * Gy[j] - delta * tt + delta * tg[u];
        const T yn = odd ? clipp(s, lo[u], hi[u]) : res_clip(s, lo[u], hi[u]);
        Gy[j] = yn;
        if constexpr (EARLY) {  // as in k_solo
          const T cq = -tg[u], tf = cq + tt;
          pri += half * yn * yn + cq * yn;
          if (!odd) {
            const T mz = __builtin_fmin(__builtin_fmax(-tf, lo[u]), hi[u]);
            dual += half * mz * mz + tf * mz;
            mx = __builtin_fmax(mx, absv(yn - mz));
          } else {
            const T mz = clipp(-tf, lo[u], hi[u]);
            dual += half * mz * mz + tf * mz;
            const T xs = yn - ((yn + cq) + tt);
            T g = maxp(absv(yn - clipp(xs, lo[u], hi[u])),
                       maxp(maxp(lo[u] - yn, zero), maxp(yn - hi[u], zero)));
            if (!finite(g)) g = inf;
            mx = __builtin_fmax(mx, g);
          }
        }
      }
    }
    __syncthreads();
    // ---- row pass: K y+, the residual, and the next d+ from K ybar = (1 + theta) K y+ -
    // theta K y (with the stop test after its verdict: the thread's own rows)
    T kn[kWideU];
    for (int s0 = wave; s0 < A.nsr; s0 += 16 * kWideU) {
      T rr[kWideU], acc[kWideU];
#pragma unroll
      for (int u = 0; u < kWideU; ++u) {
        const int i = (s0 + 16 * u) * 64 + lane;
        rr[u] = s0 + 16 * u < A.nsr && i < m ? RR[i] : zero;
      }
      wide_sums(s0, A.nsr, A.roff, A.ridx, A.rval, Gy, acc);
#pragma unroll
      for (int u = 0; u < kWideU; ++u) {
        const int i = (s0 + 16 * u) * 64 + lane;
        if (s0 + 16 * u >= A.nsr || i >= m) continue;
        const T d = Gd[i];
        const bool ineq = A.rperm[i] >= A.me;
        if constexpr (EARLY) {
          const T e = acc[u] - rr[u], w = ineq ? zero : -one;
          mx = __builtin_fmax(mx, __builtin_fmax(e, w * e));
          dual = (dual - rr[u] * d) - d * zero;
          kn[u] = acc[u];
          if (!one_group) KN[i] = acc[u];
        } else if (more) {
          T p = d + sigma_n * (((one + theta) * acc[u] - theta * KY[i]) - rr[u]);
          if (ineq) p = res_pos(p);
          Gd[i] = p;
          KY[i] = acc[u];
        }
      }
    }
    if constexpr (EARLY) {
      const T s2 = two_sums(pri, dual);
      const T wm = wave_fmax(mx);
      if ((lane & 31) == 0) red[wave * 4 + (lane >> 5)] = s2;
      if (lane == 0) red[wave * 4 + 2] = wm;
      __syncthreads();
      const T* rl = red + (lane & 15) * 4;
      const T xp = row16_combine(rl[0], OpAdd()), xd = row16_combine(rl[1], OpAdd());
      const T xm = row16_combine(rl[2], OpFMax());
      const T gap = maxp(xp - xd, zero) / maxp(one, maxp(absv(xp), absv(xd)));
      // the 64 lanes hold the four rows' identical totals in each row's lane 0
      if (__builtin_amdgcn_readfirstlane(finite(gap) && xm <= tol && gap <= tol ? 1 : 0)) {
        accepted = true;
        ++it;
        break;
      }
      auto move = [&](int s, T acc) {
        const int i = s * 64 + lane;
        if (s >= A.nsr || i >= m) return;
        T p = Gd[i] + sigma_n * (((one + theta) * acc - theta * KY[i]) - RR[i]);
        if (A.rperm[i] >= A.me) p = res_pos(p);
        Gd[i] = p;
        KY[i] = acc;
      };
      if (more && one_group) {
#pragma unroll
        for (int u = 0; u < kWideU; ++u) move(wave + 16 * u, kn[u]);
      } else if (more) {
        for (int s = wave; s < A.nsr; s += 16)
          move(s, s * 64 + lane < m ? KN[s * 64 + lane] : zero);
      }
    }
    __syncthreads();
  }
  __syncthreads();
  for (int e = t; e < n; e += 1024) A.Y[(int64_t)A.cperm[e] * Bp + b] = Gy[e];
  for (int e = t; e < m; e += 1024) A.D[(int64_t)A.rperm[e] * Bp + b] = Gd[e];
  if (EARLY && t == 0) {
    A.count[b] = (int32_t)it;
    A.done[b] = accepted ? 1 : 0;
  }
}

// ---------------------------------------------------------------------------
// The dense adapter (dense.py:85-106): rows and columns of tens of entries, so several lanes
// share each, and the loop runs until the last sample is accepted.  The streaming passes
// walked each row serially on a few wavefronts: 244 us per iteration at n = 60, m = 37,
// B = 64.  Launch 1 (FIRST) runs every sample to its own acceptance and leaves the largest
// count; launch 2 takes each sample from its state there to that count.
// ---------------------------------------------------------------------------
constexpr int kSoloDenseW = 12;

// sum over the 2^l lanes that share a row, in every one of them
template <typename T>
__device__ __forceinline__ T lane_sum(T v, int l) {
  if (l >= 1) v += dpp_move<0xB1>(v);   // lane ^ 1
  if (l >= 2) v += dpp_move<0x4E>(v);   // lane ^ 2
  if (l >= 3) v += dpp_move<0x141>(v);  // the other quad of 8
  if (l >= 4) v += dpp_move<0x140>(v);  // the other half of 16
  if (l >= 5) v += __shfl_xor(v, 16);
  if (l >= 6) v += __shfl_xor(v, 32);
  return v;
}

template <typename T>
__device__ __forceinline__ T dense_sum(const T (&v)[kSoloDenseW],
                                       const uint32_t (&ix)[kSoloDenseW / 2], int groups, int l,
                                       const unsigned char* lds) {
  const T acc = groups <= 1 ? dot_regs<4>(v, ix, lds)
                            : (groups == 2 ? dot_regs<8>(v, ix, lds) : dot_regs<12>(v, ix, lds));
  return lane_sum(acc, l);
}

template <typename T, bool FIRST, bool HELP, int MAXB>
__global__ __launch_bounds__(MAXB) void k_solo_dense(SoloDense<T> A) {
  extern __shared__ __align__(16) unsigned char lds[];
  constexpr int W = kSoloDenseW;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int NW = (blockDim.x >> 6) - (HELP ? 1 : 0), NT = NW * 64;
  const int64_t b = blockIdx.x, Bp = A.Bp;
  const int n = A.n, m = A.m;
  const int jt = t >> A.lc, gc = t & ((1 << A.lc) - 1), it_ = t >> A.lr, gr = t & ((1 << A.lr) - 1);
  const bool col = jt < n && t < NT, row = it_ < m && t < NT;
  const bool wc = col && gc == 0, wr = row && gr == 0;  // the lane that writes
  const int j = col ? jt : 0, i = row ? it_ : 0;
  if (b >= A.batch) {
    if (FIRST && wc) A.Y[(int64_t)j * Bp + b] = A.YB[(int64_t)j * Bp + b] = T(0);
    if (FIRST && wr) A.D[(int64_t)i * Bp + b] = T(0);
    return;
  }
  const T zero = T(0), one = T(1), half = T(0.5), inf = T(__builtin_inf());
  T* Gy = reinterpret_cast<T*>(lds);
  T* Gd = Gy + n + 1;
  T* red = Gd + m + 1;
  volatile int* flag = reinterpret_cast<volatile int*>(red + (HELP ? 6 * NT : 64));
  T rv[W], cv[W];
  uint32_t rx[W / 2], cx[W / 2];
  const int rs = A.rptr[i], re = row ? A.rptr[i + 1] : rs;
  const int cs = n ? A.cptr[j] : 0, ce = col ? A.cptr[j + 1] : cs;
  const int64_t vb = A.vbp > 1 ? b : 0;
#pragma unroll
  for (int k = 0; k < W; ++k) {
    const int er = rs + (k << A.lr) + gr, ec = cs + (k << A.lc) + gc;
    const bool okr = er < re, okc = ec < ce;
    rv[k] = okr ? A.RV[(int64_t)er * A.vbp + vb] : zero;
    cv[k] = okc ? A.CV[(int64_t)ec * A.vbp + vb] : zero;
    const uint32_t xr = (uint32_t)((okr ? A.ridx[er] : n) * (int)sizeof(T));
    const uint32_t xc = (uint32_t)((n + 1 + (okc ? A.cidx[ec] : m)) * (int)sizeof(T));
    if (k & 1) {
      rx[k / 2] |= xr << 16;
      cx[k / 2] |= xc << 16;
    } else {
      rx[k / 2] = xr;
      cx[k / 2] = xc;
    }
  }
  const int rgr = (A.rw + 3) >> 2, cgr = (A.cw + 3) >> 2;
  const int64_t jb = (int64_t)j * Bp + b, ib = (int64_t)i * Bp + b;
  const T q = col ? A.Q[jb] : one, cj = col ? A.C[jb] : zero;
  const T lo = col ? A.LO[jb] : zero, hi = col ? A.HI[jb] : zero;
  const T rr = row ? A.R[ib] : zero;
  T y = col ? A.Y[jb] : zero, d = row ? A.D[ib] : zero;
  const bool ineq = i >= A.me;
  T tau = res_uniform(A.step0[b]), sig = res_uniform(A.step0[Bp + b]);
  T th = res_uniform(A.accel ? A.step0[4 * Bp + b] : one);
  const T gam = res_uniform(A.gam ? A.gam[b] : one);
  T pa = one / (one + tau * q);
  auto advance = [&]() {  // the accelerated update (kernels.py:279-283)
    if (!A.accel) return;
    T g1[1] = {gam}, t1[1] = {tau}, s1[1] = {sig}, h1[1] = {th}, a1[1], d1[1];
    res_qp_schedule<T, 1>(g1, t1, s1, h1, a1, d1);
    tau = t1[0];
    sig = s1[0];
    th = h1[0];
    pa = one / (one + tau * q);
  };
  auto step = [&](T tt) -> T {  // the factored prox (kernels.py:140-142)
    return clipp(pa * ((y - tau * tt) - tau * cj), lo, hi);
  };
  if (t == 0) {
    Gy[n] = zero;
    Gd[m] = zero;
    *flag = 0;
  }

  if constexpr (!FIRST) {
    const int64_t from = A.count ? A.count[b] : 0;
    const int64_t to = A.last ? *A.last : A.iters;
    for (int64_t k = 0; k < from && A.accel; ++k) advance();
    if (wc) Gy[j] = A.YB[jb];
    if (wr) Gd[i] = d;
    __syncthreads();
    for (int64_t it = from; it < to; ++it) {
      const T acc = dense_sum(rv, rx, rgr, A.lr, lds);
      T p = d + sig * (acc - rr);
      if (ineq) p = maxp(p, zero);
      d = p;
      if (wr) Gd[i] = p;
      __syncthreads();
      const T tt = dense_sum(cv, cx, cgr, A.lc, lds);
      const T yn = step(tt);
      if (wc) Gy[j] = yn + th * (yn - y);
      y = yn;
      advance();
      __syncthreads();
    }
    if (wc) A.Y[jb] = y;
    if (wr) A.D[ib] = d;
    if (t == 0 && A.last) A.count[b] = (int32_t)to;
    return;
  }

  if (wc) Gy[j] = y;
  __syncthreads();
  T ky = dense_sum(rv, rx, rgr, A.lr, lds);
  {
    T p = d + sig * (ky - rr);
    if (ineq) p = maxp(p, zero);
    d = p;
    if (wr) Gd[i] = p;
  }
  __syncthreads();
  const T tol = A.tolv[b];
  auto judge = [&](T pri, T dual, T mx) -> bool {
    const T gap = maxp(pri - dual, zero) / maxp(one, maxp(absv(pri), absv(dual)));
    return finite(gap) && mx <= tol && gap <= tol;
  };
  if (HELP && wave == NW) {
    for (int64_t it = 0;; ++it) {
      if ((it >= 2 && __builtin_amdgcn_readfirstlane(*flag)) || it > A.iters) return;
      T pri = zero, dual = zero, mx = inf;
      if (it > 0) {
        const T* pt = red + ((it - 1) & 1) * 3 * NT + lane;
        mx = zero;
        add_parts(pt, NW, NT, pri, dual, mx);
        const T s2 = two_sums(pri, dual);
        pri = read_lane(s2, 0);
        dual = read_lane(s2, 32);
        mx = wave_fmax(mx);
      }
      __syncthreads();
      const bool ok = judge(pri, dual, mx);
      if (lane == 0) *flag = ok ? 1 : 0;
      __syncthreads();
    }
  }
  T yp = y, ypp = y, dk = d, dkp = d, th1 = one, th2 = one;
  T q_pri = zero, q_dual = zero, q_max = inf;
  int64_t it = 0;
  bool accepted = false;
  for (;; ++it) {
    if (it >= 2 && __builtin_amdgcn_readfirstlane(*flag)) {
      accepted = true;
      break;
    }
    if (it > A.iters) break;
    const bool run = it < A.iters;
    const T r_pri = q_pri, r_dual = q_dual, r_max = q_max;
    ypp = yp;
    yp = y;
    q_pri = q_dual = q_max = zero;
    if (run) {
      const T tt = dense_sum(cv, cx, cgr, A.lc, lds);
      const T yn = step(tt);
      y = yn;
      if (wc) {
        Gy[j] = yn;
        q_pri = half * q * yn * yn + cj * yn;
        const T tf = cj + tt;
        const T mz = q > T(1e-12) ? clipp(-tf / q, lo, hi) : (tf >= zero ? lo : hi);
        q_dual = half * q * (mz * mz) + tf * mz;
        T g = maxp(maxp(lo - yn, zero), maxp(yn - hi, zero));
        if (!finite(g)) g = inf;
        q_max = g;
      }
    }
    if constexpr (!HELP) {
      const T s2 = two_sums(r_pri, r_dual);
      const T mx = wave_fmax(r_max);
      if ((lane & 31) == 0) red[wave * 4 + (lane >> 5)] = s2;
      if (lane == 0) red[wave * 4 + 2] = mx;
    }
    __syncthreads();
    dkp = dk;
    dk = d;
    th2 = th1;
    th1 = th;
    const T theta = th;
    if (run) advance();
    if (run) {
      const T acc = dense_sum(rv, rx, rgr, A.lr, lds);
      if (wr) {
        const T e = acc - rr, w = ineq ? zero : -one;
        q_max = __builtin_fmax(q_max, __builtin_fmax(e, w * e));
        q_dual = (q_dual - rr * d) - d * zero;
      }
      if (it + 1 < A.iters) {
        T p = d + sig * (((one + theta) * acc - theta * ky) - rr);
        if (ineq) p = maxp(p, zero);
        d = p;
        if (wr) Gd[i] = p;
      }
      ky = acc;
    }
    if constexpr (HELP) {
      T* pt = red + (it & 1) * 3 * NT + t;
      pt[0] = q_pri;
      pt[NT] = q_dual;
      pt[2 * NT] = q_max;
    } else if (wave == NW - 1) {
      const T* rl = red + (lane & 15) * 4;
      const bool in = (lane & 15) < NW;
      const T xp = row16_combine(in ? rl[0] : zero, OpAdd());
      const T xd = row16_combine(in ? rl[1] : zero, OpAdd());
      const T mx = row16_combine(in ? rl[2] : zero, OpFMax());
      const bool ok = it > 0 && judge(xp, xd, mx);
      if (lane == 0) *flag = ok ? 1 : 0;
    }
    __syncthreads();
  }
  if (accepted) {  // the state of iteration it - 2, and its ybar
    if (wc) A.YB[jb] = yp + th2 * (yp - ypp);
    y = yp;
    dk = dkp;
  }
  if (wc) A.Y[jb] = y;
  if (wr) A.D[ib] = dk;
  if (t == 0) {
    const int32_t k = (int32_t)(accepted ? it - 1 : A.iters);
    A.count[b] = k;
    A.done[b] = accepted ? 1 : 0;
    atomicMax(A.last, k);
  }
}

int rest_entries(const purin_cp_plan* p, int W) {
  int k = 0;
  for (int w : p->sl_rw) k += rest_of(w, W) * 64;
  for (int w : p->sl_cw) k += rest_of(w, W) * 64;
  return k;
}

constexpr size_t kLdsMax = 160 * 1024;

int solo_waves(const purin_cp_plan* p) { return std::max(p->sl_nsr, p->sl_nsc); }

int cu_count(const purin_cp_plan* p) {
  int cus = 0;
  return hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, p->device) == hipSuccess
             ? cus
             : 256;
}

// The workgroup: wavefronts of rows and columns (with idle ones) and whether one more
// runs the stop test.
struct SoloBlock {
  int waves;
  bool help;
};

// A CU holds 16 wavefronts of these kernels (fp64).  The wavefront of the stop test pays
// wherever it costs no workgroup per CU, and in a launch of one round: us per iteration at
// B = 256 without / with it 1.32 / 0.71 (n = 60), 1.25 / 1.03 (n = 500), 1.68 / 1.4 (n =
// 950), at B = 8192 10.9 / 18.7 with four wavefronts (four workgroups per CU against three),
// 23.7 / 30.3 with eight (two against one).  Five to seven become eight, which
// spreads over the four SIMDs alike: six (n = 310) took 31 us at B = 8192, eight 18.5.
SoloBlock solo_block(const purin_cp_plan* p, int64_t batch, bool early) {
  const int w = solo_waves(p);
  if (!early) return {w > 4 && w < 8 ? 8 : w, false};
  if (w > 15) return {w, false};
  const int64_t cus = cu_count(p);
  if ((w == 4 && batch > 2 * cus) || (w == 8 && batch > cus)) return {w, false};
  return {w > 3 && w < 8 ? 7 : w, true};
}

// LDS of the larger of the two loops (with the stop test)
size_t solo_lds(const purin_cp_plan* p, SoloBlock k) {
  const size_t es = elem_size(p);
  const size_t parts = k.help ? 6 * 64 * (size_t)k.waves : 64;
  return (size_t)(p->n + 1 + p->m + 1 + parts + 2) * es + (size_t)rest_entries(p, kSoloW) * (es + 2);
}

template <typename T, int MODE>
int launch_mode(hipStream_t st, const Solo<T>& A, SoloBlock k, size_t lds, bool early) {
  auto kern = !early ? k_solo<T, kSoloW, MODE, false, false>
                     : (k.help ? k_solo<T, kSoloW, MODE, true, true>
                               : k_solo<T, kSoloW, MODE, true, false>);
  if (int rc = raise_lds_cap((const void*)kern, lds)) return rc;
  kern<<<(unsigned)A.Bp, 64u * (unsigned)(k.waves + (k.help ? 1 : 0)), lds, st>>>(A);
  return PURIN_CP_OK;
}

}  // namespace

// Against the tile kernels (two fp64 or eight fp32 samples per workgroup, one workgroup per
// CU), us per iteration with the stop test / without:
//   fp64  n = 60, B = 256: 0.71 / 0.37 (tile 2.09 / 0.67); n = 500, B = 8192: 23.7 / 9.3
//         (37.9 / 13.5); n = 800: 38.1 / 17.0 (39.3 / 14.1); n = 1020: 49.0 / 19.6 (40.8 / 16.7)
//   fp32  n = 250, B = 8192: 6.5 / 2.5 (16.1 / 4.3); n = 500: 13.5 / 6.4 (16.4 / 4.6);
//         n = 800: 32.3 / 15.5 (17.7 / 4.7), B = 512: 2.0 / 1.0 (4.2 / 1.2)
// so a sample per workgroup while its wavefronts leave a CU at least two of them, and above
// that for the batches of the first rounds.  Rows and columns past the registers (``chain``
// entries of the widest) take LDS, and with it workgroups from a CU, and a workgroup's time
// grows with them while the tiles' stream is shared by their samples (us per iteration, stop
// test / without, here against the tiles):
//   fp64  one workgroup per CU: n = 200, a dense row: B = 256 4.2 / 3.7 (5.6 / 4.3), B = 1024
//         22.4 / 15.0 (11.2 / 8.7); n = 500, rows of 40: B = 512 4.8 / 3.5 (3.4 / 2.1)
//         two: n = 250, rows of 40, B = 2048 9.3 / 7.1 (11.2 / 6.8); n = 120, a dense row,
//         B = 8192 43.4 / 38.9 (63.1 / 44.8)
//         n = 700, B = 2048: rows of 12 9.7 (9.9), of 24 11.3 (10.8), of 40 16.0 (13.2)
//   fp32  n = 240, a dense row (one per CU): B = 256 4.3 / 4.2 (9.7 / 7.4), B = 1024 17.9 / 16.4
//         (9.7 / 7.5); n = 300, five rows of 150 (two): B = 1024 6.5 / 6.1 (7.3 / 5.1),
//         B = 8192 51.7 (28.9); n = 400, rows of 40 (three): B = 1024 3.8 / 3.4 (4.8 / 2.7),
//         B = 2048 6.2 (4.9); n = 250, rows of 12: B = 1024 1.4 / 0.9 (4.0 / 1.3), B = 2048 2.6 /
//         1.7 (4.0 / 1.2); n = 500, rows of 24, B = 2048: 5.2 (4.7)
// A full round of the fp32 tiles is 2048 samples.  Per-sample coefficients stay in registers
// and LDS here and stream from HBM there, whatever the batch (n = 200, a dense row, B = 8192:
// fp64 186 / 118 against 202 / 151).
bool solo_fits(const purin_cp_plan* p, int64_t batch, bool early, bool values) {
  if (!p->sl_ok || p->n > kSoloMax || p->m > kSoloMax) return false;
  const size_t lds = solo_lds(p, solo_block(p, batch, early));
  if (lds > kLdsMax) return false;
  const int w = solo_waves(p);
  const int64_t cus = cu_count(p), per_cu = (int64_t)(kLdsMax / lds);
  auto past = [](const std::vector<int32_t>& v) { return v.empty() ? 0 : rest_of(v[0], kSoloW); };
  const int chain = past(p->sl_rw) + past(p->sl_cw);
  if (values) return true;
  if (p->dtype == PURIN_CP_F64) {
    if (batch <= cus) return true;
    if (w > 8) return early && w <= 13 && chain <= 16;
    return per_cu >= (early || w <= 2 ? 2 : 3);
  }
  if (early) {
    if (w > 8) return batch <= 3 * cus;
    if (per_cu >= 4 && (w < 8 || chain <= 8)) return true;
    return batch <= 2 * std::min<int64_t>(per_cu, 2) * cus;
  }
  if (chain <= 3) return w <= 4 || batch <= (w <= 8 ? 4 : 2) * cus;
  if (w <= 2 && per_cu >= 3) return true;
  return batch <= (per_cu == 1 ? 1 : (w <= 4 ? 4 : 2)) * cus;
}

template <typename T>
int solo_launch(hipStream_t st, const purin_cp_plan* p, const Solo<T>& A, int mode, bool early) {
  const SoloBlock k = solo_block(p, A.batch, early);
  const size_t lds = solo_lds(p, k);
  switch (mode) {
    case kSoloShared: return launch_mode<T, kSoloShared>(st, A, k, lds, early);
    case kSoloValues: return launch_mode<T, kSoloValues>(st, A, k, lds, early);
    default: return launch_mode<T, kSoloQP>(st, A, k, lds, early);
  }
}

static size_t wide_lds(const purin_cp_plan* p, bool early) {
  const int64_t vectors = early && p->sl_nsr > 16 * kWideU ? 3 : 2;  // d, K y (and K y+)
  return (size_t)(p->n + 1 + 1 + vectors * p->m + 64) * elem_size(p);
}

// Problems beyond the tile kernels.  us per iteration with the stop test / without, against
// the streaming passes: n = 12001 (flow, m = 3001) fp32 13.4 / 9.9 at B = 64 (107 / 23.5),
// 55.9 / 40.1 at B = 1024 (162 / 59.8); n = 6000, m = 2100 fp64 12.6 / 10.1 (85.6 / 17.9) and
// 51.4 / 40.5 (140 / 59.1).  Fixed iterations of more than 4096 rows stay on the passes,
// whose narrow column tiles serve them.
bool solo_wide_holds(const purin_cp_plan* p) {
  return !p->res_ok && !p->diag && p->m >= 1 && wide_lds(p, false) <= kLdsMax;
}
bool solo_wide_can(const purin_cp_plan* p, bool early) {
  if (!p->sl_ok || !solo_wide_holds(p)) return false;
  if (!early && p->sl_nsr > 16 * kWideU) return false;
  return wide_lds(p, early) <= kLdsMax;
}

// Every workgroup streams the matrix, and a CU holds one; the passes read it once per 128
// (fp64) or 256 (fp32) samples.  us per iteration here against the passes, n = 8000:
//   a row or column far longer than a wavefront's share of the entries is one wavefront's
//   chain, in every round of the launch: fp64 a dense row fixed B = 256 949 (1526), B = 512
//   1897 (1606), stop test B = 512 1953 (2932), B = 1024 3900 (3183); a column of 3000 fixed
//   B = 512 694 (932), B = 1024 1412 (1041); four rows of 2000 fixed B = 512 465 (579), B =
//   1024 933 (614), stop test B = 4096 4071 (4488)
//   even rows, fixed: fp64 up to 400 wide (800,000 entries) even or better from B = 256 on,
//   but B = 64 rows of 200 135 (119), n = 12000 rows of 75 107 (81); fp32 rows of 50 324 (392)
//   at B = 4096, of 100 162 (136) at B = 1024, n = 6000 rows of 300 1116 (668) at B = 4096;
//   up to B = 512 better at any width.  With the stop test better at any width and batch.
//   fp32, few rows and columns, fixed: a round is latency, n = 4200, m = 200 B = 1024 14.8
//   (18.5), B = 4096 58.9 (47.3); n = 5000, m = 400 B = 4096 70 (60); m = 1500 80 (93).
bool solo_wide_fits(const purin_cp_plan* p, int64_t batch, bool early) {
  if (!solo_wide_can(p, early)) return false;
  const int64_t cus = cu_count(p), chain = (int64_t)p->sl_rw[0] + p->sl_cw[0];
  const bool uneven = chain > std::max<int64_t>(128, 4 * ((p->sl_rn + p->sl_cn) / kWideThreads));
  if (early) return !uneven || chain <= 2048 || batch <= 2 * cus;
  if (uneven) return batch <= (chain <= 4096 ? 2 : 1) * cus;
  if (p->dtype == PURIN_CP_F64) return p->nnz <= 160000 || batch > 128;
  if (batch > 4 * cus && p->n + p->m < 5500) return false;
  return batch <= 2 * cus || p->nnz <= 13 * (p->n + p->m);
}

template <typename T>
int solo_wide_launch(hipStream_t st, const purin_cp_plan* p, const SoloWide<T>& A, bool early) {
  const size_t lds = wide_lds(p, early);
  auto kern = early ? k_solo_wide<T, true> : k_solo_wide<T, false>;
  if (int rc = raise_lds_cap((const void*)kern, lds)) return rc;
  kern<<<(unsigned)A.Bp, kWideThreads, lds, st>>>(A);
  return PURIN_CP_OK;
}
template int solo_wide_launch<double>(hipStream_t, const purin_cp_plan*, const SoloWide<double>&, bool);
template int solo_wide_launch<float>(hipStream_t, const purin_cp_plan*, const SoloWide<float>&, bool);

// Lanes per row (log2) and entries per lane for rows of up to ``width`` entries.
static void dense_lanes(int width, int* l, int* entries) {
  *l = 0;
  while (*l < 6 && (width + (1 << *l) - 1) >> *l > kSoloDenseW) ++*l;
  *entries = (width + (1 << *l) - 1) >> *l;
}

bool solo_dense_fits(const purin_cp_plan* p) {
  if (!p->sl_ok || p->n > kSoloMax || p->m > kSoloMax || p->m < 1) return false;
  int lr, lc, rw, cw;
  dense_lanes(p->sl_rw[0], &lr, &rw);
  dense_lanes(p->sl_cw[0], &lc, &cw);
  return rw <= kSoloDenseW && cw <= kSoloDenseW && p->m << lr <= 1024 && p->n << lc <= 1024;
}

template <typename T>
int solo_dense_launch(hipStream_t st, const purin_cp_plan* p, SoloDense<T> A, bool early) {
  dense_lanes(p->sl_rw[0], &A.lr, &A.rw);
  dense_lanes(p->sl_cw[0], &A.lc, &A.cw);
  const int waves = (int)((std::max<int64_t>(p->m << A.lr, p->n << A.lc) + 63) / 64);
  const size_t lds = (size_t)(p->n + 1 + p->m + 1 + 6 * 64 * waves + 2) * sizeof(T);
  if (early) {  // up to 512 threads the kernel has registers to spare (above, fp64 spills 128 B)
    auto kern = waves < 8 ? k_solo_dense<T, true, true, 512>
                          : (waves < 16 ? k_solo_dense<T, true, true, 1024>
                                        : k_solo_dense<T, true, false, 1024>);
    if (int rc = raise_lds_cap((const void*)kern, lds)) return rc;
    kern<<<(unsigned)A.Bp, 64u * (unsigned)(waves + (waves < 16 ? 1 : 0)), lds, st>>>(A);
  } else {
    A.count = A.last = nullptr;
  }
  if (int rc = raise_lds_cap((const void*)k_solo_dense<T, false, false, 1024>, lds)) return rc;
  k_solo_dense<T, false, false, 1024><<<(unsigned)A.Bp, 64u * (unsigned)waves, lds, st>>>(A);
  return PURIN_CP_OK;
}
template int solo_dense_launch<double>(hipStream_t, const purin_cp_plan*, SoloDense<double>, bool);
template int solo_dense_launch<float>(hipStream_t, const purin_cp_plan*, SoloDense<float>, bool);

template int solo_launch<double>(hipStream_t, const purin_cp_plan*, const Solo<double>&, int, bool);
template int solo_launch<float>(hipStream_t, const purin_cp_plan*, const Solo<float>&, int, bool);

}  // namespace purin
