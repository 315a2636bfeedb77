// Restarted GMRES of the implicit VJP, one workgroup per sample.
//
// Reference: _batched_restarted_gmres
// (src/purin/solvers/primal_dual_interior_point/operators.py:792-1125).  The
// samples are independent within a restart cycle, so a workgroup runs a whole
// cycle of one sample: operator, both projections, the Givens step and the stop
// test of every Arnoldi step, then the correction and the candidate's residual.
// The batch meets only between cycles, where the reference bounds a cycle by the
// iterations left (the longest sample's steps count, Gmr::ctrl).
//
// The batch-minor passes this replaces took about a dozen dependent launches per
// Arnoldi step, each over the whole batch: ~110 us a step for a small problem
// whatever its bytes, and with a large one every sample's basis was streamed until
// the slowest sample stopped.  Here a step costs its own sample's work.
//
// The basis is raw, as in adjoint.hip (k_gm_tri): slot i holds Z_i, the image of
// step i - 1 after one projection, v_j = sum_{i <= j} Z_i Tm[i][j], so a step reads
// the prefix twice.  The dot pass walks the elements last to first and the update
// pass first to last, so the update begins on rows the caches still hold.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "gmres.hpp"

namespace purin {

namespace {

constexpr int kLd = kGmrRestart + 1;  // row stride of the per-sample triangular matrices

// --- reductions over a wavefront ------------------------------------------------

template <typename T>
struct Words;
template <>
struct Words<double> {
  static constexpr int N = 2;
};
template <>
struct Words<float> {
  static constexpr int N = 1;
};

// a', b' = [a's lower half, b's lower half], [a's upper half, b's upper half] of
// the wavefront (BIT = 32) or of each half wavefront's pair of rows (BIT = 16): the
// sum a' + b' leaves a's total over the pair in the lower and b's in the upper half.
template <int BIT, typename T>
__device__ __forceinline__ T swap_add(T a, T b) {
  constexpr int N = Words<T>::N;
  typedef uint32_t U __attribute__((ext_vector_type(N)));
  U x = __builtin_bit_cast(U, a), y = __builtin_bit_cast(U, b);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    if constexpr (BIT == 32) {
      const auto r = __builtin_amdgcn_permlane32_swap(x[i], y[i], false, false);
      x[i] = r[0];
      y[i] = r[1];
    } else {
      const auto r = __builtin_amdgcn_permlane16_swap(x[i], y[i], false, false);
      x[i] = r[0];
      y[i] = r[1];
    }
  }
  return __builtin_bit_cast(T, x) + __builtin_bit_cast(T, y);
}

// v of the lane that DPP control CTRL pairs with this one
template <int CTRL, typename T>
__device__ __forceinline__ T dpp(T v) {
  constexpr int N = Words<T>::N;
  typedef int U __attribute__((ext_vector_type(N)));
  U x = __builtin_bit_cast(U, v);
#pragma unroll
  for (int i = 0; i < N; ++i) x[i] = __builtin_amdgcn_update_dpp(0, x[i], CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(T, x);
}
constexpr int kMirror16 = 0x140;  // lane i of a row of 16 with lane 15 - i
constexpr int kMirror8 = 0x141;   // lane i of a half row with lane 7 - i
constexpr int kMirror4 = 0x1b;    // lane i of a quad with lane 3 - i
constexpr int kMirror2 = 0xb1;    // lane i of a pair with lane 1 - i

// one halving step on lane bit BIT: lanes with the bit keep the upper half of v
template <int BIT, int N, typename T>
__device__ __forceinline__ void halve(T (&v)[kGmrRestart], int lane) {
  constexpr int H = N / 2;
#pragma unroll
  for (int i = 0; i < H; ++i) {
    if constexpr (BIT >= 16) {
      v[i] = swap_add<BIT>(v[i], v[i + H]);
    } else {
      constexpr int C = BIT == 8 ? kMirror16 : (BIT == 4 ? kMirror8 : kMirror4);
      const bool up = (lane & BIT) != 0;
      const T send = up ? v[i] : v[i + H];
      const T keep = up ? v[i + H] : v[i];
      v[i] = keep + dpp<C>(send);
    }
  }
}

// plain sums over the remaining lane bits below and including BIT
template <int BIT, typename T>
__device__ __forceinline__ T fold(T v) {
  if constexpr (BIT >= 32) v = swap_add<32>(v, v);
  if constexpr (BIT >= 16) v = swap_add<16>(v, v);
  if constexpr (BIT >= 8) v = v + dpp<kMirror16>(v);
  if constexpr (BIT >= 4) v = v + dpp<kMirror8>(v);
  if constexpr (BIT >= 2) v = v + dpp<kMirror4>(v);
  return v + dpp<kMirror2>(v);
}

// Sums of v[0..N) over the wavefront (N = 4, 8, 16 or 32): lane l returns the sum
// of v[l * N / 64].  A butterfly that halves the values held at each step: 31
// exchanges for 32 sums in place of 6 each.
template <int N, typename T>
__device__ __forceinline__ T wave_sums(T (&v)[kGmrRestart], int lane) {
  if constexpr (N == 32) {
    halve<32, 32>(v, lane);
    halve<16, 16>(v, lane);
    halve<8, 8>(v, lane);
    halve<4, 4>(v, lane);
    halve<2, 2>(v, lane);
    return v[0] + dpp<kMirror2>(v[0]);
  } else if constexpr (N == 16) {
    halve<32, 16>(v, lane);
    halve<16, 8>(v, lane);
    halve<8, 4>(v, lane);
    halve<4, 2>(v, lane);
    return fold<2>(v[0]);
  } else if constexpr (N == 8) {
    halve<32, 8>(v, lane);
    halve<16, 4>(v, lane);
    halve<8, 2>(v, lane);
    return fold<4>(v[0]);
  } else {
    halve<32, 4>(v, lane);
    halve<16, 2>(v, lane);
    return fold<8>(v[0]);
  }
}

// the value every lane holds, as a scalar
template <typename T>
__device__ __forceinline__ T uniform(T v) {
  constexpr int N = Words<T>::N;
  typedef int U __attribute__((ext_vector_type(N)));
  U x = __builtin_bit_cast(U, v);
#pragma unroll
  for (int i = 0; i < N; ++i) x[i] = __builtin_amdgcn_readfirstlane(x[i]);
  return __builtin_bit_cast(T, x);
}

// LDS written by one lane of a wavefront is read by another after this
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The sum of v over lanes l and l ^ 32, in both
template <typename T>
__device__ __forceinline__ T both_halves(T v) {
  return swap_add<32>(v, v);
}

// v of lane l (wave-uniform l), as a scalar
template <typename T>
__device__ __forceinline__ T lane_value(T v, int l) {
  constexpr int N = Words<T>::N;
  typedef int U __attribute__((ext_vector_type(N)));
  U x = __builtin_bit_cast(U, v);
#pragma unroll
  for (int i = 0; i < N; ++i) x[i] = __builtin_amdgcn_readlane(x[i], l);
  return __builtin_bit_cast(T, x);
}

// --- LDS of one workgroup ---------------------------------------------------------

// Elements: u [n + 1], w [m + 1], the wavefronts' partial sums [BS / 64][33], shares of
// slices [BS], then per-sample algebra (below), then the basis where it fits.
constexpr int kAlg = 3 * kLd * kLd + 9 * kLd;

template <typename T>
struct Alg {  // pointers into the algebra block
  T *Tm, *Hu, *H, *P, *Gv, *Q, *U2, *G1, *Cs, *Sn, *g, *Wc;
  __device__ explicit Alg(T* p) {
    Tm = p;                 // [i][j], upper triangular
    Hu = Tm + kLd * kLd;    // unrotated Hessenberg matrix
    H = Hu + kLd * kLd;     // rotated
    P = H + kLd * kLd;
    Gv = P + kLd;
    Q = Gv + kLd;
    U2 = Q + kLd;
    G1 = U2 + kLd;
    Cs = G1 + kLd;
    Sn = Cs + kLd;
    g = Sn + kLd;
    Wc = g + kLd;
  }
};

inline size_t lds_elems(int64_t n, int64_t m, int64_t W, int restart, int bs, bool basis) {
  return (size_t)(n + 1 + m + 1 + (bs / 64) * kLd + bs + kAlg + (basis ? (restart + 1) * W : 0));
}

// --- the operator -----------------------------------------------------------------

// put(s, sum) of every slice by one wavefront: the products of its entries with x.  With
// parts > 1 (a multiple of few wide slices) that many wavefronts take every parts-th entry
// and meet in LDS: 60 serial loads of a dense row are 6 us otherwise.
template <typename T, int BS, typename Put>
__device__ __forceinline__ void slices(int ns, int parts, const int32_t* __restrict__ off,
                                       const uint16_t* __restrict__ idx, const T* __restrict__ val,
                                       const T* x, T* share, Put put) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (parts <= 1) {
    for (int s = wave; s < ns; s += BS / 64) {
      const int o0 = off[s], o1 = off[s + 1];
      T acc = T(0);
#pragma unroll 4
      for (int o = o0 + lane; o < o1; o += 64) acc += val[o] * x[idx[o]];
      put(s, acc);
    }
    return;
  }
  const int s = wave / parts, part = wave % parts;  // ns * parts <= wavefronts
  T acc = T(0);
  if (s < ns) {
    const int o0 = off[s], o1 = off[s + 1];
#pragma unroll 4
    for (int o = o0 + part * 64 + lane; o < o1; o += parts * 64) acc += val[o] * x[idx[o]];
    share[wave * 64 + lane] = acc;
  }
  __syncthreads();
  if (s < ns && part == 0) {
    for (int k = 1; k < parts; ++k) acc += share[(wave + k) * 64 + lane];
    put(s, acc);
  }
}

// out = v sc - pullback(v sc) (adjoint.hip's k_op_*): u = C (gy + 2 gb),
// w = D (gd - delta K u), out = (gy - (a u - gb), gd - w, gb - sigma K^T w).  One
// thread per row / column of a slice; u and w meet in LDS.
template <typename T, int BS, bool DG>
__device__ __forceinline__ void apply(const Gmr<T>& A, int64_t b, const T* __restrict__ v, T sc,
                                      T* __restrict__ out, T* u, T* w, T* share) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = A.n, m = A.m;
  const T* __restrict__ mask = A.mask + (size_t)b * (n + m);
  const T* __restrict__ av = DG ? A.av + (size_t)b * n : nullptr;
  const T* __restrict__ dv = DG ? A.dv + (size_t)b * n : nullptr;
  const T* __restrict__ sv = DG ? A.sv + (size_t)b * m : nullptr;
  for (int j = tid; j < n; j += BS) {
    const T gy = v[j] * sc, gb = v[n + m + j] * sc;
    const T uj = mask[j] * (gy + T(2) * gb);
    u[j] = DG ? dv[j] * uj : uj;
    out[j] = gy - ((DG ? av[j] : A.a) * uj - gb);
  }
  __syncthreads();
  const T* __restrict__ rval = A.rval + (size_t)b * A.rstride;
  slices<T, BS>(A.nsr, A.rparts, A.roff, A.ridx, rval, u, share, [&](int s, T acc) {
    const int i = s * 64 + lane;
    if (i < m) {
      const T gd = v[n + i] * sc;
      const T wi = mask[n + i] * (DG ? gd - acc : gd - A.delta * acc);
      w[i] = DG ? sv[i] * wi : wi;
      out[n + i] = gd - wi;
    }
  });
  __syncthreads();
  const T* __restrict__ cval = A.cval + (size_t)b * A.cstride;
  slices<T, BS>(A.nsc, A.cparts, A.coff, A.cidx, cval, w, share, [&](int s, T acc) {
    const int j = s * 64 + lane;
    if (j < n) {
      const T gb = v[n + m + j] * sc;
      out[n + m + j] = DG ? gb - acc : gb - A.sigma * acc;
    }
  });
  __syncthreads();
}

// --- the two passes over the prefix -------------------------------------------------

// Element e of the first nv vectors of Z into z (the last one again for i >= nv).
// One 32-bit byte offset walks the vectors from Z's scalar base, so the prefix costs
// no address registers; NV - 4 < nv <= NV.
template <typename T, int NV>
__device__ __forceinline__ void load_prefix(const T* Z, uint32_t ldb, int nv, int e, T (&z)[NV]) {
  uint32_t off = (uint32_t)e * (uint32_t)sizeof(T);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (i > 0) off += (i <= NV - 4 || i < nv) ? ldb : 0u;
    z[i] = *reinterpret_cast<const T*>(reinterpret_cast<const char*>(Z) + off);
  }
}

// red[wave][i] = the wavefront's part of Z_i . y, i < nv
template <typename T, int BS, int NV>
__device__ __forceinline__ void pass_dots(const T* Z, uint32_t ldb, int nv, const T* y, int W,
                                          T* red) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  T acc[kGmrRestart];
#pragma unroll
  for (int i = 0; i < kGmrRestart; ++i) acc[i] = T(0);
  for (int e = tid + (W - 1 - tid) / BS * BS; e >= 0 && tid < W; e -= BS) {
    const T ye = y[e];
    T z[NV];
    load_prefix<T, NV>(Z, ldb, nv, e, z);
#pragma unroll
    for (int i = 0; i < NV; ++i) acc[i] += z[i] * ye;
  }
  constexpr int N = NV <= 4 ? 4 : (NV <= 8 ? 8 : (NV <= 16 ? 16 : 32));
  const T s = wave_sums<N>(acc, lane);
  constexpr int per = 64 / N;
  if (lane % per == 0) red[wave * kLd + lane / per] = s;
}

// y <- y - sum_i q_i Z_i; red[wave][i] = the wavefront's part of Z_i . y for
// i < nv, red[wave][kLd - 1] its part of y . y
template <typename T, int BS, int NV>
__device__ __forceinline__ void pass_update(const T* Z, uint32_t ldb, int nv, T* y, int W,
                                            const T* Q, T* red) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  T acc[kGmrRestart], q[NV], nrm = T(0);
#pragma unroll
  for (int i = 0; i < kGmrRestart; ++i) acc[i] = T(0);
#pragma unroll
  for (int i = 0; i < NV; ++i) q[i] = i < nv ? uniform(Q[i]) : T(0);
  for (int e = tid; e < W; e += BS) {
    T ye = y[e];
    T z[NV];
    load_prefix<T, NV>(Z, ldb, nv, e, z);
#pragma unroll
    for (int i = 0; i < NV; ++i) ye -= q[i] * z[i];
    y[e] = ye;
#pragma unroll
    for (int i = 0; i < NV; ++i) acc[i] += z[i] * ye;
    nrm += ye * ye;
  }
  constexpr int N = NV <= 4 ? 4 : (NV <= 8 ? 8 : (NV <= 16 ? 16 : 32));
  const T s = wave_sums<N>(acc, lane);
  nrm = fold<32>(nrm);
  constexpr int per = 64 / N;
  if (lane % per == 0) red[wave * kLd + lane / per] = s;
  if (lane == 0) red[wave * kLd + kLd - 1] = nrm;
}

template <typename T, int BS, bool UPDATE>
__device__ __forceinline__ void pass(const T* Z, uint32_t ldb, int nv, T* y, int W, const T* Q,
                                     T* red) {
  // the bucket sets the registers a thread holds and the loads it has in flight
  auto go = [&](auto k) {
    constexpr int NV = decltype(k)::value;
    if constexpr (UPDATE)
      pass_update<T, BS, NV>(Z, ldb, nv, y, W, Q, red);
    else
      pass_dots<T, BS, NV>(Z, ldb, nv, y, W, red);
  };
  switch ((nv - 1) >> 2) {
    case 0: go(std::integral_constant<int, 4>{}); break;
    case 1: go(std::integral_constant<int, 8>{}); break;
    case 2: go(std::integral_constant<int, 12>{}); break;
    case 3: go(std::integral_constant<int, 16>{}); break;
    case 4: go(std::integral_constant<int, 20>{}); break;
    case 5: go(std::integral_constant<int, 24>{}); break;
    case 6: go(std::integral_constant<int, 28>{}); break;
    default: go(std::integral_constant<int, 32>{}); break;
  }
}

// --- one restart cycle --------------------------------------------------------------

template <typename T, int BS, bool DG, bool ZL>
__global__ __launch_bounds__(BS) void k_gmr_cycle(Gmr<T> A, int c, int64_t base, int64_t max_it) {
  extern __shared__ __align__(16) unsigned char gmr_raw[];
  constexpr int NW = BS / 64;
  const int64_t b = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = A.n, m = A.m, W = A.W, R = A.restart;
  int64_t done = base;
  for (int k = 0; k < c; ++k) done += A.ctrl[k];
  const int limit = (int)(max_it - done < R ? max_it - done : R);
  const T thr = A.thr[b];
  if (limit <= 0 || !(A.rinf[b] > thr)) return;  // the same for the whole workgroup
  T* u = reinterpret_cast<T*>(gmr_raw);
  T* w = u + n + 1;
  T* red = w + m + 1;
  T* share = red + NW * kLd;
  const Alg<T> S(share + BS);
  T* zl = S.Wc + kLd;
  __shared__ T s_inv;
  __shared__ int s_on;
  T* __restrict__ X = A.X + (size_t)b * A.Wp;
  T* __restrict__ Rr = A.R + (size_t)b * A.Wp;
  const T* __restrict__ G = A.G + (size_t)b * A.Wp;
  T* Z = ZL ? zl : A.Z + (size_t)b * (R + 1) * A.Wp;
  const int64_t ld = ZL ? W : A.Wp;
  const uint32_t ldb = (uint32_t)(ld * sizeof(T));
  const T eps = T(1e-30), brk = T(1e-14);

  // beta = ||r||, Z_0 = r / max(beta, eps)
  T acc = T(0);
  for (int e = tid; e < W; e += BS) acc += Rr[e] * Rr[e];
  acc = fold<32>(acc);
  if (lane == 0) red[wave * kLd] = acc;
  if (tid == 0) {
    u[n] = T(0);
    w[m] = T(0);
  }
  __syncthreads();
  T beta = T(0);
#pragma unroll
  for (int k = 0; k < NW; ++k) beta += red[k * kLd];
  beta = __builtin_sqrt(beta);
  const T scale = T(1) / maxp(beta, eps);
  for (int e = tid; e < W; e += BS) Z[e] = Rr[e] * scale;
  if (tid < kLd) {
    S.g[tid] = tid == 0 ? beta : T(0);
    S.U2[tid] = T(0);
  }
  if (tid == 0) {
    S.Tm[0] = T(1);
    s_inv = T(1);
    s_on = 1;
  }
  __syncthreads();

  int it = 0;
  while (it < limit) {
    const int nv = it + 1;
    T* y = Z + (int64_t)nv * ld;
    apply<T, BS, DG>(A, b, Z + (int64_t)it * ld, s_inv, y, u, w, share);
    pass<T, BS, false>(Z, ldb, nv, y, W, S.Q, red);
    __syncthreads();
    // The algebra runs on one wavefront: lanes j and j + 32 share vector j's sums (even
    // and odd terms), which halves their chains of LDS reads.
    const int vj = lane & 31, half = lane >> 5;
    if (wave == 0) {  // p = Z^T y; g1 = Tm^T p; q1 = Tm g1
      if (lane < nv) {
        T s = T(0);
#pragma unroll
        for (int k = 0; k < NW; ++k) s += red[k * kLd + lane];
        S.P[lane] = s;
      }
      wave_sync();
      T s = T(0);
      if (vj < nv) {
#pragma unroll 8
        for (int i = half; i <= vj; i += 2) s += S.Tm[i * kLd + vj] * S.P[i];
      }
      s = both_halves(s);
      if (lane < nv) S.G1[lane] = s;
      wave_sync();
      s = T(0);
      if (vj < nv) {
#pragma unroll 8
        for (int j = vj + half; j < nv; j += 2) s += S.Tm[vj * kLd + j] * S.G1[j];
      }
      s = both_halves(s);
      if (lane < nv) S.Q[lane] = s;
    }
    __syncthreads();
    pass<T, BS, true>(Z, ldb, nv, y, W, S.Q, red);
    __syncthreads();
    if (wave == 0) {  // the step's algebra (k_gm_tri, MODE 2)
      if (lane < nv || lane == kLd - 1) {
        T s = T(0);
#pragma unroll
        for (int k = 0; k < NW; ++k) s += red[k * kLd + lane];
        S.P[lane] = s;
      }
      wave_sync();
      T g2 = T(0), cj = T(0);
      if (vj < nv) {
#pragma unroll 8
        for (int i = half; i <= vj; i += 2) g2 += S.Tm[i * kLd + vj] * S.P[i];
#pragma unroll 8
        for (int k = (vj > 0 ? vj - 1 : 0) + half; k < it; k += 2)
          cj += S.Hu[vj * kLd + k] * S.U2[k];
      }
      g2 = both_halves(g2);
      cj = both_halves(cj);
      T col = T(0), rc_ = T(0), rs_ = T(0);
      if (lane < nv) {
        S.Gv[lane] = g2;
        col = (S.G1[lane] + g2) - cj;
        S.Hu[lane * kLd + it] = col;
        rc_ = S.Cs[lane];
        rs_ = S.Sn[lane];
      }
      wave_sync();
      const T ss = fold<32>(lane < nv ? g2 * g2 : T(0));
      const T n1 = S.P[kLd - 1];
      const T d2 = n1 - ss;
      const T next_norm = d2 < T(0) ? T(0) : __builtin_sqrt(d2);  // NaN stays NaN
      // the rotations of the earlier steps, in order, on every lane alike, from the
      // registers of the lanes that hold them
      T carry = lane_value(col, 0), hcol = T(0);
      for (int ri = 0; ri < it; ++ri) {
        const T cc = lane_value(rc_, ri), sn = lane_value(rs_, ri), nx = lane_value(col, ri + 1);
        const T h = cc * carry + sn * nx;
        hcol = lane == ri ? h : hcol;
        carry = -sn * carry + cc * nx;
      }
      if (lane < it) S.H[lane * kLd + it] = hcol;
      const T rnorm = hypotv(carry, next_norm);
      const T safe = maxp(rnorm, eps);
      const T nc = rnorm > eps ? carry / safe : T(1);
      const T ns = rnorm > eps ? next_norm / safe : T(0);
      const T pc = S.g[it], pn = S.g[it + 1];
      const T rc = nc * pc + ns * pn, rn = -ns * pc + nc * pn;
      const T inv = T(1) / maxp(next_norm, eps);
      const T est = absv(rn);
      const bool on = finite(est) && finite(rnorm) && finite(n1) && !(next_norm <= brk) && est > thr;
      // column it + 1 of Tm: v_{it+1} = (Z_{it+1} - Z Tm g2) / nu, and u = g2 / nu
      T tc = T(0);
      if (vj < nv) {
#pragma unroll 8
        for (int j = vj + half; j < nv; j += 2) tc += S.Tm[vj * kLd + j] * S.Gv[j];
      }
      tc = both_halves(tc);
      wave_sync();
      if (lane < nv) {
        S.Tm[lane * kLd + nv] = -(tc * inv);
        S.U2[lane] = g2 * inv;
      }
      if (lane == 0) {
        S.Hu[nv * kLd + it] = next_norm;
        S.Cs[it] = nc;
        S.Sn[it] = ns;
        S.H[it * kLd + it] = rnorm;
        S.g[it] = rc;
        S.g[nv] = rn;
        S.Tm[nv * kLd + nv] = inv;
        s_inv = inv;
        s_on = on ? 1 : 0;
      }
    }
    __syncthreads();
    ++it;
    if (!s_on) break;
  }
  // back substitution (operators.py:902-917) and Wc = Tm coeff, so that
  // x += sum_j coeff_j v_j = sum_i Wc_i Z_i
  if (wave == 0) {
    T num = lane < it ? S.g[lane] : T(0);
    for (int row = it - 1; row >= 0; --row) {
      const T d = S.H[row * kLd + row];
      if (lane == row) S.Gv[row] = num / (absv(d) > eps ? d : T(1));
      wave_sync();
      if (lane < row) num -= S.H[lane * kLd + row] * S.Gv[row];
    }
    wave_sync();
    if (lane < it) {
      T s = T(0);
#pragma unroll 8
      for (int j = lane; j < it; ++j) s += S.Tm[lane * kLd + j] * S.Gv[j];
      S.Wc[lane] = s;
    }
  }
  __syncthreads();
  int fin = 1;
  for (int e = tid; e < W; e += BS) {
    T s = T(0);
#pragma unroll 8
    for (int i = 0; i < it; ++i) s += S.Wc[i] * Z[(int64_t)i * ld + e];
    const T x = X[e] + s;
    X[e] = x;
    if (!finite(x)) fin = 0;
  }
  __syncthreads();
  // the candidate's residual r = g - A x (operators.py:1084-1091); the basis is free
  apply<T, BS, DG>(A, b, X, T(1), Z, u, w, share);
  T big = T(0);
  for (int e = tid; e < W; e += BS) {
    const T r = G[e] - Z[e];
    Rr[e] = r;
    big = maxp(big, absv(r));
  }
#pragma unroll
  for (int h = 32; h > 0; h >>= 1) {
    big = maxp(big, __shfl_xor(big, h));
    fin &= __shfl_xor(fin, h);
  }
  if (lane == 0) {
    red[wave * kLd] = big;
    red[wave * kLd + 1] = fin ? T(1) : T(0);
  }
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int k = 1; k < NW; ++k) {
      big = maxp(big, red[k * kLd]);
      fin &= red[k * kLd + 1] != T(0) ? 1 : 0;
    }
    A.rinf[b] = big;
    A.xfin[b] = fin ? T(1) : T(0);
    A.total[b] += it;
    atomicMax(&A.ctrl[c], it);
  }
}

// --- BiCGSTAB over the batch --------------------------------------------------------

// The batch's sums of the workgroups' N values: each leaves its own in ``part``, and the
// last to arrive adds them and hands them to ``then`` (one thread).  The order is fixed,
// whichever arrives last: samples tid, tid + BS, ... in each thread, the lanes' tree, then the
// wavefronts in order.
template <typename T, int BS, int N, typename Then>
__device__ __forceinline__ void batch_sums(const GmrBi<T>& B, T (&v)[N], T* red, Then then) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int NW = BS / 64;
  __shared__ int s_last;
  auto block = [&](T (&x)[N]) {  // sums over the workgroup, in thread 0
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const T s = fold<32>(x[k]);
      if (lane == 0) red[wave * kLd + k] = s;
    }
    __syncthreads();
    if (tid == 0) {
#pragma unroll
      for (int k = 0; k < N; ++k) {
        x[k] = red[k];
        for (int w = 1; w < NW; ++w) x[k] += red[w * kLd + k];
      }
    }
    __syncthreads();
  };
  block(v);
  if (tid == 0) {
#pragma unroll
    for (int k = 0; k < N; ++k) B.part[k * B.batch + blockIdx.x] = v[k];
    __threadfence();
    s_last = atomicAdd(B.ticket, 1) == (int)gridDim.x - 1;
  }
  __syncthreads();
  if (!s_last) return;
  __threadfence();
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] = T(0);
  for (int64_t b = tid; b < B.batch; b += BS) {
#pragma unroll
    for (int k = 0; k < N; ++k)
      v[k] += __hip_atomic_load(&B.part[k * B.batch + b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  block(v);
  if (tid == 0) {
    *B.ticket = 0;
    then(v);
  }
}

// The LDS of the products: u [n + 1], w [m + 1], partial sums, shares of slices.
template <typename T, int BS>
struct BiLds {
  T *u, *w, *red, *share;
  __device__ BiLds(unsigned char* raw, int n, int m) {
    u = reinterpret_cast<T*>(raw);
    w = u + n + 1;
    red = w + m + 1;
    share = red + (BS / 64) * kLd;
    if (threadIdx.x == 0) {
      u[n] = T(0);
      w[m] = T(0);
    }
  }
};

// scalars for the next iteration: rho_ = rhat . r, beta, and whether it runs
template <typename T>
__device__ __forceinline__ void bi_next(const GmrBi<T>& B, T rs, T rho) {
  T* sc = B.sc;
  sc[kBiRhoN] = rho;
  sc[kBiBeta] = rho / sc[kBiRho] * sc[kBiAlpha] / sc[kBiOmega];
  sc[kBiGo] = rs > sc[kBiAtol2] && sc[kBiK] < (T)B.max_iterations && sc[kBiK] >= T(0) ? T(1) : T(0);
}

// rhat = p = q = r0 = b; rho = alpha = omega = 1
template <typename T, int BS>
__global__ __launch_bounds__(BS) void k_bic_start(Gmr<T> A, GmrBi<T> B) {
  extern __shared__ __align__(16) unsigned char gmr_raw[];
  const BiLds<T, BS> S(gmr_raw, A.n, A.m);
  const T* g = A.G + (size_t)blockIdx.x * A.Wp;
  T* Z = A.Z + (size_t)blockIdx.x * (A.restart + 1) * A.Wp;
  T v[1] = {T(0)};
  for (int e = threadIdx.x; e < A.W; e += BS) {
    const T x = g[e];
    Z[e] = Z[A.Wp + e] = Z[2 * A.Wp + e] = x;
    v[0] += x * x;
  }
  batch_sums<T, BS, 1>(B, v, S.red, [&](T (&t)[1]) {
    T* sc = B.sc;
    sc[kBiBS] = t[0];
    sc[kBiAtol2] = maxp(B.tol * B.tol * t[0], B.atol * B.atol);
    sc[kBiRho] = sc[kBiAlpha] = sc[kBiOmega] = T(1);
    sc[kBiK] = sc[kBiIt] = T(0);
    bi_next(B, t[0], t[0]);
  });
}

// p = r + beta (p - omega q), q = A p, alpha = rho / (rhat . q)
template <typename T, int BS>
__global__ __launch_bounds__(BS) void k_bic_p(Gmr<T> A, GmrBi<T> B) {
  extern __shared__ __align__(16) unsigned char gmr_raw[];
  if (B.sc[kBiGo] == T(0)) return;
  const BiLds<T, BS> S(gmr_raw, A.n, A.m);
  const int64_t b = blockIdx.x;
  const T* R = A.R + (size_t)b * A.Wp;
  T* Z = A.Z + (size_t)b * (A.restart + 1) * A.Wp;
  T *P = Z + A.Wp, *Q = Z + 2 * A.Wp;
  const T beta = B.sc[kBiBeta], omega = B.sc[kBiOmega];
  for (int e = threadIdx.x; e < A.W; e += BS) P[e] = R[e] + beta * (P[e] - omega * Q[e]);
  __syncthreads();
  apply<T, BS, true>(A, b, P, T(1), Q, S.u, S.w, S.share);
  T v[1] = {T(0)};
  for (int e = threadIdx.x; e < A.W; e += BS) v[0] += Z[e] * Q[e];
  batch_sums<T, BS, 1>(B, v, S.red, [&](T (&t)[1]) { B.sc[kBiAlphaN] = B.sc[kBiRhoN] / t[0]; });
}

// s = r - alpha q, t = A s, omega = (t . s) / (t . t)
template <typename T, int BS>
__global__ __launch_bounds__(BS) void k_bic_s(Gmr<T> A, GmrBi<T> B) {
  extern __shared__ __align__(16) unsigned char gmr_raw[];
  if (B.sc[kBiGo] == T(0)) return;
  const BiLds<T, BS> S(gmr_raw, A.n, A.m);
  const int64_t b = blockIdx.x;
  const T* R = A.R + (size_t)b * A.Wp;
  T* Z = A.Z + (size_t)b * (A.restart + 1) * A.Wp;
  T *Q = Z + 2 * A.Wp, *Sv = Z + 3 * A.Wp, *Tv = Z + 4 * A.Wp;
  const T alpha = B.sc[kBiAlphaN];
  for (int e = threadIdx.x; e < A.W; e += BS) Sv[e] = R[e] - alpha * Q[e];
  __syncthreads();
  apply<T, BS, true>(A, b, Sv, T(1), Tv, S.u, S.w, S.share);
  T v[3] = {T(0), T(0), T(0)};
  for (int e = threadIdx.x; e < A.W; e += BS) {
    const T s = Sv[e], t = Tv[e];
    v[0] += s * s;
    v[1] += t * s;
    v[2] += t * t;
  }
  batch_sums<T, BS, 3>(B, v, S.red, [&](T (&t)[3]) {
    B.sc[kBiSS] = t[0];
    B.sc[kBiOmegaN] = t[1] / t[2];
  });
}

// x and r, with the early exit; the iteration's end and the next one's scalars
template <typename T, int BS>
__global__ __launch_bounds__(BS) void k_bic_x(Gmr<T> A, GmrBi<T> B) {
  extern __shared__ __align__(16) unsigned char gmr_raw[];
  if (B.sc[kBiGo] == T(0)) return;
  const BiLds<T, BS> S(gmr_raw, A.n, A.m);
  const int64_t b = blockIdx.x;
  T* X = A.X + (size_t)b * A.Wp;
  T* R = A.R + (size_t)b * A.Wp;
  const T* Z = A.Z + (size_t)b * (A.restart + 1) * A.Wp;
  const T *P = Z + A.Wp, *Sv = Z + 3 * A.Wp, *Tv = Z + 4 * A.Wp;
  const T alpha = B.sc[kBiAlphaN], omega = B.sc[kBiOmegaN];
  const bool early = B.sc[kBiSS] < B.sc[kBiAtol2];
  T v[2] = {T(0), T(0)};
  for (int e = threadIdx.x; e < A.W; e += BS) {
    const T s = Sv[e];
    const T r = early ? s : s - omega * Tv[e];
    X[e] = early ? X[e] + alpha * P[e] : X[e] + (alpha * P[e] + omega * s);
    R[e] = r;
    v[0] += r * r;
    v[1] += Z[e] * r;
  }
  batch_sums<T, BS, 2>(B, v, S.red, [&](T (&t)[2]) {
    T* sc = B.sc;
    T k = (sc[kBiOmegaN] == T(0) || sc[kBiAlphaN] == T(0)) ? T(-11) : sc[kBiK] + T(1);
    if (sc[kBiRhoN] == T(0)) k = T(-10);
    sc[kBiK] = k;
    sc[kBiIt] += T(1);
    sc[kBiRho] = sc[kBiRhoN];
    sc[kBiAlpha] = sc[kBiAlphaN];
    sc[kBiOmega] = sc[kBiOmegaN];
    bi_next(B, t[0], t[1]);
  });
}

constexpr size_t kLdsMax = 160 * 1024;

template <typename T, int BS, bool DG, bool ZL>
int launch(hipStream_t st, const Gmr<T>& A, int64_t batch, int c, int64_t base, int64_t max_it) {
  const size_t lds = lds_elems(A.n, A.m, A.W, A.restart, BS, ZL) * sizeof(T);
  if (int rc = raise_lds_cap((const void*)k_gmr_cycle<T, BS, DG, ZL>, lds)) return rc;
  k_gmr_cycle<T, BS, DG, ZL><<<(unsigned)batch, BS, lds, st>>>(A, c, base, max_it);
  return PURIN_CP_OK;
}

template <typename T, bool DG>
int dispatch(hipStream_t st, const Gmr<T>& A, int64_t batch, int c, int64_t base, int64_t max_it) {
  // Small problems keep the basis in LDS too (half the LDS, so that two workgroups
  // share a CU), with 4 wavefronts, the smallest (two elements a lane) with one:
  // 20,000 samples of W = 38 took 2.5 ms with four.
  if (A.W <= 128) return launch<T, 64, DG, true>(st, A, batch, c, base, max_it);
  if (A.W <= 512 && lds_elems(A.n, A.m, A.W, A.restart, 256, true) * sizeof(T) <= kLdsMax / 2)
    return launch<T, 256, DG, true>(st, A, batch, c, base, max_it);
  if (A.W <= 512) return launch<T, 256, DG, false>(st, A, batch, c, base, max_it);
  return launch<T, 512, DG, false>(st, A, batch, c, base, max_it);
}

}  // namespace

bool gmr_holds(const purin_cp_plan* p) {
  return lds_elems(p->n, p->m, 0, 0, 512, false) * elem_size(p) + 64 <= kLdsMax;
}

// BiCGSTAB's sums over the batch go through one counter and the last workgroup: ms per call
// here against the passes, n = 60: B = 1024 5.3 (6.3), B = 2048 8.7 (6.9), B = 4096 18.0 (8.0).
//
// GMRES: each sample stops by itself here, so whole calls are faster at any batch (ms, fp64:
// n = 64 B = 16384 5.9 (11.7); n = 300 43 (71), with rows of 24 37.6 (39.5)), except where a
// long row or column is one wavefront's chain, ``chain`` entries, in every round of the launch
// and not small beside the vectors, whose streams hide it where two workgroups share a CU:
//   fp64  n = 600, chain 400: B = 1024 18.2 (20.8), B = 2048 34.6 (27.9)
//         n = 1000, chain 1000: B = 1024 29.6 (35.4), B = 2048 56.7 (46.8)
//         n = 4000, chain 2000: B = 512 66 (78), B = 1024 123 (99)
//         n = 8000, chain 8000: B = 512 194 (225), B = 1024 366 (269)
//         but n = 2000, chain 600, B = 8192 193 (216); n = 4000, chain 1150, B = 4096 202 (217)
//         one workgroup per CU, n = 8000, m = 2500, chain 1500: B = 512 89 (102), B = 2048 343 (248)
//   fp32  n = 600, chain 400: B = 4096 21.9 (28.6)
//         chain 600, coefficients per sample: B = 2048 29.5 (32.3), B = 4096 51.4 (42.6)
//         n = 4000, chain 2000: B = 1024 55 (79), B = 4096 189 (148)
//         n = 8000, chain 8000: B = 1024 256 (223)
int64_t gmr_batch(const purin_cp_plan* p, int64_t restart, bool dense) {
  if (!p->sl_ok || restart > kGmrRestart || !gmr_holds(p)) return 0;
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, p->device) != hipSuccess)
    cus = 256;
  if (dense) return 4 * (int64_t)cus;
  const int64_t W = 2 * p->n + p->m;
  auto longest = [&](const std::vector<int32_t>& w) -> int64_t {
    return w.empty() ? 0 : w[0] / gmr_parts(W, (int)w.size(), w[0]);
  };
  const int64_t chain = longest(p->sl_rw) + longest(p->sl_cw);
  const size_t lds = lds_elems(p->n, p->m, 0, 0, 512, false) * elem_size(p);
  if (chain <= std::max<int64_t>(128, lds <= kLdsMax / 2 ? W / 7 : W / 50)) return INT64_MAX;
  if (p->dtype == PURIN_CP_F64) return (chain <= 256 ? 8 : (chain <= 1024 ? 4 : 2)) * (int64_t)cus;
  return (chain <= 512 ? 16 : (chain <= 1024 ? 8 : (chain <= 4096 ? 4 : 2))) * (int64_t)cus;
}

template <typename T>
int gmr_cycle(hipStream_t st, const Gmr<T>& A, int64_t batch, bool dg, int c, int64_t base,
              int64_t max_iterations) {
  return dg ? dispatch<T, true>(st, A, batch, c, base, max_iterations)
            : dispatch<T, false>(st, A, batch, c, base, max_iterations);
}

int gmr_parts(int64_t W, int slices, int widest) {
  const int waves = W <= 128 ? 1 : (W <= 512 ? 4 : 8);
  return slices > 0 && widest >= 16 ? std::max(1, waves / slices) : 1;
}

template <typename T>
int gmr_bicgstab(hipStream_t st, const Gmr<T>& A, const GmrBi<T>& B, int iterations, bool start) {
  auto go = [&](auto bs) -> int {
    constexpr int BS = decltype(bs)::value;
    const size_t lds = lds_elems(A.n, A.m, 0, 0, BS, false) * sizeof(T);
    for (const void* k : {(const void*)k_bic_start<T, BS>, (const void*)k_bic_p<T, BS>,
                          (const void*)k_bic_s<T, BS>, (const void*)k_bic_x<T, BS>})
      if (int rc = raise_lds_cap(k, lds)) return rc;
    const unsigned g = (unsigned)B.batch;
    if (start) k_bic_start<T, BS><<<g, BS, lds, st>>>(A, B);
    for (int k = 0; k < iterations; ++k) {
      k_bic_p<T, BS><<<g, BS, lds, st>>>(A, B);
      k_bic_s<T, BS><<<g, BS, lds, st>>>(A, B);
      k_bic_x<T, BS><<<g, BS, lds, st>>>(A, B);
    }
    return PURIN_CP_OK;
  };
  return A.W <= 512 ? go(std::integral_constant<int, 256>{}) : go(std::integral_constant<int, 512>{});
}
template int gmr_bicgstab<double>(hipStream_t, const Gmr<double>&, const GmrBi<double>&, int, bool);
template int gmr_bicgstab<float>(hipStream_t, const Gmr<float>&, const GmrBi<float>&, int, bool);

template int gmr_cycle<double>(hipStream_t, const Gmr<double>&, int64_t, bool, int, int64_t, int64_t);
template int gmr_cycle<float>(hipStream_t, const Gmr<float>&, int64_t, bool, int, int64_t, int64_t);

}  // namespace purin
