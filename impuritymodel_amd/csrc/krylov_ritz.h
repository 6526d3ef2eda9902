// Ritz pairs of a Lanczos tridiagonal on one workgroup: eigenvalues by Sturm
// multisection, vectors by inverse iteration.
#pragma once

#include "common.h"

namespace imped {

constexpr int MAX_NEV = 16;

__device__ __forceinline__ uint64_t splitmix(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

__device__ __forceinline__ double u01(uint64_t x) { return (double)(splitmix(x) >> 11) * (1.0 / 9007199254740992.0); }

// 1/x to within an ulp: the hardware reciprocal estimate refined by two
// Newton steps (a short dependent chain, where a correctly rounded division
// is a long one).
__device__ __forceinline__ double rcp_nr(double x) {
  double r = __builtin_amdgcn_rcp(x);
  double e = fma(-x, r, 1.0);
  r = fma(r, e, r);
  e = fma(-x, r, 1.0);
  return fma(r, e, r);
}

// Sturm counts at P shifts from the leading principal minors of T - x:
// d_0 = 1, d_1 = a_0 - x, d_{i+1} = (a_i - x) d_i - b_{i-1}^2 d_{i-1}; the
// number of eigenvalues of the m x m tridiagonal (a, b) below x is the
// number of sign changes in d_0, ..., d_m.  There is no division, so the
// dependent chain of a step is one FMA (the quotient form d_i / d_{i-1}
// needs a reciprocal per step); the P recurrences are interleaved.  Every 8
// steps the pair (d_{i-1}, d_i) is scaled by the power of two that brings
// the larger to [0.5, 1): exact, so no sign or ratio changes, and within 8
// steps the minors grow or shrink by at most (1 + |a - x| + b^2)^8 or b^16,
// far from the exponent range.  A minor that is exactly zero counts by its
// sign bit: its neighbours have opposite signs (b != 0 inside the chain), so
// the two changes around it count one either way.
template <int P>
__device__ __forceinline__ void sturm_counts(const double* a, const double* b, int m, const double* x, int* cnt) {
  double d0[P], d1[P];  // d_{i-1}, d_i
#pragma unroll
  for (int p = 0; p < P; ++p) {
    d0[p] = 1.0;
    d1[p] = a[0] - x[p];
    cnt[p] = (int)((unsigned)__double2hiint(d1[p]) >> 31);
  }
  auto step = [&](int i) {
    const double ai = a[i], bb = b[i - 1] * b[i - 1];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const double dn = fma(ai - x[p], d1[p], -bb * d0[p]);
      cnt[p] += (int)((unsigned)(__double2hiint(dn) ^ __double2hiint(d1[p])) >> 31);
      d0[p] = d1[p];
      d1[p] = dn;
    }
  };
  int i = 1;
  for (; i + 8 <= m; i += 8) {
#pragma unroll
    for (int u = 0; u < 8; ++u) step(i + u);
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int e = max(__builtin_amdgcn_frexp_exp(d0[p]), __builtin_amdgcn_frexp_exp(d1[p]));
      d0[p] = __builtin_amdgcn_ldexp(d0[p], -e);
      d1[p] = __builtin_amdgcn_ldexp(d1[p], -e);
    }
  }
  for (; i < m; ++i) step(i);
}

// Inverse iteration for the eigenvector of (a, b) at lambda; LU with partial
// pivoting of the shifted tridiagonal.  y and work (4m + m ints) are
// thread-private (LDS or global).  Every recurrence carries its running
// values in registers, so no iteration waits on a store it just made.
__device__ __forceinline__ void tri_inverse_iteration(const double* __restrict__ a, const double* __restrict__ b, int m, double lambda,
                                      double* __restrict__ y, double* __restrict__ dd, double* __restrict__ uu,
                                      double* __restrict__ ww, double* __restrict__ ll, int* __restrict__ piv,
                                      uint64_t seed) {
  double scale = 0.0;
#pragma unroll 8
  for (int i = 0; i < m; ++i) scale = fmax(scale, fabs(a[i]) + (i < m - 1 ? fabs(b[i]) : 0.0));
  const double tiny = 2.2e-16 * (scale > 0 ? scale : 1.0);
  // (d, u): diagonal and superdiagonal of the current row after elimination
  double d = a[0] - lambda, u = m > 1 ? b[0] : 0.0;
#pragma unroll 8
  for (int i = 0; i < m - 1; ++i) {
    const double sub = b[i];
    const double dn = a[i + 1] - lambda;
    const double un = i + 1 < m - 1 ? b[i + 1] : 0.0;
    // rows i and i+1 interchanged when |d| < |sub|; both cases by selects
    // (the lanes of different eigenvalues choose differently, and branches
    // would run both cases one after the other), one reciprocal
    const bool sw = !(fabs(d) >= fabs(sub));
    const double pv = sw ? sub : (d == 0.0 ? tiny : d);
    const double mult = (sw ? d : sub) * rcp_nr(pv);
    dd[i] = pv;
    uu[i] = sw ? dn : u;
    ww[i] = sw ? un : 0.0;
    ll[i] = mult;
    piv[i] = sw ? 1 : 0;
    const double d_keep = dn - mult * u, d_swap = u - mult * dn;
    const double u_swap = -mult * un;
    d = sw ? d_swap : d_keep;
    u = sw ? u_swap : un;
  }
  if (d == 0.0) d = tiny;
  dd[m - 1] = d;
  uu[m - 1] = 0.0;
  ww[m - 1] = 0.0;
  // back substitution multiplies by the guarded reciprocal pivots
#pragma unroll 8
  for (int i = 0; i < m; ++i) {
    double dv = dd[i];
    if (fabs(dv) < tiny) dv = dv < 0 ? -tiny : tiny;
    dd[i] = rcp_nr(dv);
  }
#pragma unroll 8
  for (int i = 0; i < m; ++i) y[i] = 0.5 + u01(seed + (uint64_t)i);
  for (int it = 0; it < 3; ++it) {
    // forward: L^-1 with the interchanges; yi is the running y[i]
    double yi = y[0];
#pragma unroll 8
    for (int i = 0; i < m - 1; ++i) {
      const double y1 = y[i + 1];
      const bool sw = piv[i] != 0;
      const double top = sw ? y1 : yi, bot = sw ? yi : y1;
      y[i] = top;
      yi = bot - ll[i] * top;
    }
    y[m - 1] = yi;
    // back substitution with U (bandwidth 3); y1, y2 = y[i+1], y[i+2]
    double y1 = 0.0, y2 = 0.0, nrm = 0.0;
#pragma unroll 8
    for (int i = m - 1; i >= 0; --i) {
      double r = y[i];
      if (i + 1 < m) r -= uu[i] * y1;
      if (i + 2 < m) r -= ww[i] * y2;
      const double v = r * dd[i];
      y[i] = v;
      nrm += v * v;
      y2 = y1;
      y1 = v;
    }
    const double inv = 1.0 / sqrt(nrm);
#pragma unroll 8
    for (int i = 0; i < m; ++i) y[i] *= inv;
  }
}

struct EigenArgs {
  const int64_t* row_base;
  const int64_t* chain_n;
  const int64_t* rowptr;
  const int32_t* col;
  const double2* val;
  int nev;
  int max_steps;
  double tol;
  uint64_t seed;
  void* vstore;        // per chain: msteps(c) * n vectors (double or double2), offset voff[c]
  const int64_t* voff;
  void* wbuf;          // per chain: n at row_base
  double2* coef;       // per chain: max_steps
  double* ab;          // per chain: 2*max_steps (alpha then beta)
  double* yk;          // per chain: nev*max_steps
  double* tw;          // per chain: nev * 5 * max_steps
  int* tpiv;           // per chain: nev * max_steps
  double* evals;
  double2* evecs;
  int32_t* steps;
  int32_t* conv;
  const int32_t* chain_list;
  int dgks;          // 1: second Gram-Schmidt pass only when needed
  int check_every;   // Ritz check interval (steps)
  int check_start;   // no check before this many steps (except at the last step)
  int lstride;       // LDS arrays: Gram-Schmidt coefficients (lstride + 2), then, when lds_work = 1,
  int lds_work;      //   alpha/beta (2 lstride), per eigenvalue y (lstride), LU work (4 lstride) and
                     //   pivots (lstride ints); lstride >= every chain's steps
  int kl;            // register kernels: vectors kept in LDS per group of waves
  int nmax;          //   and rows of the launch's largest chain
};

// Lowest nev eigenvalues of the symmetric tridiagonal (a, b) of size m by
// multisection: the workgroup's first `points` threads split into nev groups; each
// evaluates Sturm counts at G interior points of its interval per round and keeps
// the sub-interval where the count crosses k, shrinking it G+1 times per round.
// The values' last bits depend on `points` alone, not on BT.
// hint (or null): the same eigenvalues of a leading block of (a, b).  By
// Cauchy interlacing they bound the new ones from above, so a first round of
// points hint - scale 10^(-16 r / (G-2)) (r < G-1) and hint + 1e-14 scale
// brackets each new value within about its distance from the hint, and the
// ordinary rounds start from that bracket (the Gershgorin interval when the
// hint does not bracket it).
template <int BT>
__device__ __forceinline__ void ritz_values(const double* a, const double* b, int m, int nev, const double* hint, double* s_lam,
                            double* s_lo, double* s_hi, int* s_first, int* s_flag, int points = BT) {
  __shared__ double s_part[3][BT / 64];
  __shared__ double s_bounds[3];
  {
    double lo = INFINITY, hi = -INFINITY, sc = 0.0;
    for (int i = threadIdx.x; i < m; i += BT) {
      const double r = (i > 0 ? fabs(b[i - 1]) : 0.0) + (i < m - 1 ? fabs(b[i]) : 0.0);
      lo = fmin(lo, a[i] - r);
      hi = fmax(hi, a[i] + r);
      sc = fmax(sc, fabs(a[i]) + r);
    }
    for (int off = 32; off > 0; off >>= 1) {
      lo = fmin(lo, __shfl_xor(lo, off));
      hi = fmax(hi, __shfl_xor(hi, off));
      sc = fmax(sc, __shfl_xor(sc, off));
    }
    if ((threadIdx.x & 63) == 0) {
      s_part[0][threadIdx.x >> 6] = lo;
      s_part[1][threadIdx.x >> 6] = hi;
      s_part[2][threadIdx.x >> 6] = sc;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int wv = 1; wv < BT / 64; ++wv) {
        lo = fmin(lo, s_part[0][wv]);
        hi = fmax(hi, s_part[1][wv]);
        sc = fmax(sc, s_part[2][wv]);
      }
      s_bounds[0] = lo - 1e-14 * sc - 1e-300;
      s_bounds[1] = hi + 1e-14 * sc + 1e-300;
      s_bounds[2] = sc;
    }
  }
  __syncthreads();
  const int G = points / nev;
  const int g = threadIdx.x / G, r = threadIdx.x % G;
  const double scale = s_bounds[2];
  if ((int)threadIdx.x < nev) {
    s_lo[threadIdx.x] = s_bounds[0];
    s_hi[threadIdx.x] = s_bounds[1];
  }
  if (hint != nullptr) {
    auto hint_point = [&](int k, int rr) {
      return rr < G - 1 ? hint[k] - scale * exp10(-16.0 * (double)rr / (double)(G - 2)) : hint[k] + 1e-14 * scale;
    };
    if ((int)threadIdx.x < nev) s_first[threadIdx.x] = G;
    __syncthreads();
    if (g < nev) {
      double x = hint_point(g, r);
      int cnt;
      sturm_counts<1>(a, b, m, &x, &cnt);
      if (cnt > g) atomicMin(&s_first[g], r);
    }
    __syncthreads();
    if ((int)threadIdx.x < nev) {
      const int k = threadIdx.x, f = s_first[k];
      if (f < G) {  // otherwise the hint does not bound the value: Gershgorin interval
        if (f > 0) s_lo[k] = fmax(s_lo[k], hint_point(k, f - 1));
        s_hi[k] = fmin(s_hi[k], hint_point(k, f));
      }
    }
  }
  __syncthreads();
  for (int round = 0; round < 64; ++round) {
    if ((int)threadIdx.x < nev) s_first[threadIdx.x] = G;
    if (threadIdx.x == 0) *s_flag = 0;
    __syncthreads();
    if (g < nev) {
      const double lo = s_lo[g], hi = s_hi[g];
      double x = lo + (hi - lo) * (double)(r + 1) / (double)(G + 1);
      int cnt;
      sturm_counts<1>(a, b, m, &x, &cnt);
      if (cnt > g) atomicMin(&s_first[g], r);
    }
    __syncthreads();
    if ((int)threadIdx.x < nev) {
      const int k = threadIdx.x;
      const double lo = s_lo[k], hi = s_hi[k];
      const int f = s_first[k];
      const double nlo = f == 0 ? lo : lo + (hi - lo) * (double)f / (double)(G + 1);
      const double nhi = f == G ? hi : lo + (hi - lo) * (double)(f + 1) / (double)(G + 1);
      s_lo[k] = nlo;
      s_hi[k] = nhi;
      const double mid = 0.5 * (nlo + nhi);
      if (nhi - nlo > 2.2e-16 * fmax(fabs(nlo), fabs(nhi)) + 1e-300 && mid > nlo && mid < nhi) atomicOr(s_flag, 1);
    }
    __syncthreads();
    if (*s_flag == 0) break;
    __syncthreads();
  }
  if ((int)threadIdx.x < nev) s_lam[threadIdx.x] = 0.5 * (s_lo[threadIdx.x] + s_hi[threadIdx.x]);
  __syncthreads();
}

// Orthonormalize the inverse-iteration vectors of clustered eigenvalues
// (|lam_k - lam_q| <= 1e-3 max(1, |lam_k|)) in order, by wave 0 of the
// workgroup (lane-parallel dot products and updates).
__device__ __forceinline__ void ortho_clustered(double* Y, int ys, int m, int ne, const double* lam) {
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x;
  for (int k = 1; k < ne; ++k) {
    double* yk = Y + (size_t)k * ys;
    for (int q = 0; q < k; ++q) {
      if (fabs(lam[k] - lam[q]) > 1e-3 * fmax(1.0, fabs(lam[k]))) continue;
      const double* yq = Y + (size_t)q * ys;
      double d = 0.0;
      for (int i = lane; i < m; i += 64) d += yq[i] * yk[i];
      d = wave_sum(d);
      double nn = 0.0;
      for (int i = lane; i < m; i += 64) {
        yk[i] -= d * yq[i];
        nn += yk[i] * yk[i];
      }
      const double inv = 1.0 / sqrt(wave_sum(nn));
      for (int i = lane; i < m; i += 64) yk[i] *= inv;
    }
  }
}

}  // namespace imped
