// eigen_reg_kernel and its launch for one element type (krylov_reg.h);
// eigen_reg_real.hip and eigen_reg_cplx.hip instantiate it.
#pragma once

#include <algorithm>

#include "krylov_reg_dev.h"
#include "krylov_ritz.h"

namespace imped {

namespace {

// Lowest eigenpairs of one chain per workgroup, the Krylov basis in registers
// (krylov_reg.h): start vector, recurrence, Gram-Schmidt rule, Ritz checks and
// outcome of eigen_kernel.  T = double when H is real.
//
// What bounds it: as the Lanczos kernel, the dependent sequence of a step; the
// checks (Sturm multisection, inverse iteration on one lane per pair) are a
// further 20 to 75 us a chain.  Measured on one MI355X, launch time before (basis
// in LDS or memory, 8 waves per chain) -> now: 4096 complex chains of 90 and 100
// rows 15.4 -> 4.1 ms, 194 of them 0.53 -> 0.43 ms, 2 of them 0.52 -> 0.40 ms; one
// real chain of 190 rows 0.78 -> 0.56 ms.
template <int NQ, int G, int R, class T>
__global__ __launch_bounds__(64 * NQ * G, 2) void eigen_reg_kernel(EigenArgs a) {
  constexpr int BT = 64 * NQ * G;
  using Basis = RegBasis<NQ, G, R, T>;
  __shared__ int s_done, s_full, s_flag;
  __shared__ double s_lam[MAX_NEV], s_lo[MAX_NEV], s_hi[MAX_NEV];
  __shared__ double s_hint[MAX_NEV];  // Ritz values of the previous check
  __shared__ int s_first[MAX_NEV];
  extern __shared__ double2 lds[];
  const int c = a.chain_list[blockIdx.x];
  const int n = (int)a.chain_n[c];
  const int64_t base = a.row_base[c];
  const int nev = a.nev;
  if (n == 0) {
    if (threadIdx.x == 0) {
      a.steps[c] = 0;
      a.conv[c] = 1;
    }
    return;
  }
  const int mmax = a.max_steps < n ? a.max_steps : n;
  // Sturm points by the chain's size: every instance that may hold it has the threads
  const int points = n <= 64 ? 64 : 256;
  // LDS: tridiagonal and Ritz work arrays (stride L), the residual, the basis
  const int L = a.lstride;
  double* sa = reinterpret_cast<double*>(lds);
  double* sb = sa + L;
  double* Y = sb + L;
  double* twb = Y + (size_t)nev * L;
  int* pivb = reinterpret_cast<int*>(twb + (size_t)nev * 4 * L);
  double* p0 = twb + (size_t)nev * 4 * L + ((size_t)nev * L + 1) / 2;
  p0 += (p0 - sa) & 1;
  T* xs = reinterpret_cast<T*>(p0);
  Basis b;
  b.init(n, mmax, a.kl, p0 + ((size_t)a.nmax * Basis::D + 1) / 2 * 2, reinterpret_cast<T*>(a.vstore) + a.voff[c]);
  RegRows<NQ * G, G, R, T> h;
  h.load(a.rowptr + base, a.col, a.val, b.g, b.row, b.on);
  // seeded random start vector (real when T is real)
  T w[R], vp[R];
  double p = 0.0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint64_t u = a.seed * 0x100000001B3ull + (uint64_t)c * 0x9E3779B97F4A7C15ull + 2 * (uint64_t)b.row[r];
    const double xr = b.on[r] ? u01(u) - 0.5 : 0.0;
    const double xi = reg_real_v<T> || !b.on[r] ? 0.0 : u01(u + 1) - 0.5;
    set1(w[r], xr, xi);
    set1(vp[r], 0.0, 0.0);
    p = add_re(p, w[r], w[r]);
  }
  auto publish = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (b.g == 0 && b.on[r]) xs[b.row[r]] = w[r];
  };
  publish();
  double sc = 1.0 / sqrt(b.row_sum(p, 1)), bprev = 0.0;
  int m = 0, converged = 0, hint_ne = -1;
  // no Ritz check before min(check_start, n/2) steps (the last step is always checked)
  const int cstart = a.check_start < n / 2 ? a.check_start : n / 2;
  // eigen_kernel's check of T_m (beta_m = bt): true when the chain is done
  auto ritz_check = [&](bool last, double bt) __attribute__((always_inline)) -> bool {
    const int ne = nev < m ? nev : m;
    const bool have_prev = ne == hint_ne;
    ritz_values<BT>(sa, sb, m, ne, have_prev ? s_hint : nullptr, s_lam, s_lo, s_hi, s_first, &s_flag, points);
    // the vectors are formed only once no Ritz value moved by more than tol
    // max(1, |lam|) since the previous check
    if (threadIdx.x == 0) s_full = (last || have_prev) ? 1 : 0;
    __syncthreads();
    if (!last && have_prev && (int)threadIdx.x < ne &&
        !(fabs(s_lam[threadIdx.x] - s_hint[threadIdx.x]) <= a.tol * fmax(1.0, fabs(s_lam[threadIdx.x]))))
      atomicAnd(&s_full, 0);
    __syncthreads();
    if ((int)threadIdx.x < ne) s_hint[threadIdx.x] = s_lam[threadIdx.x];
    hint_ne = ne;
    if (threadIdx.x == 0) s_done = 1;
    __syncthreads();
    if (s_full) {
      if ((int)threadIdx.x < nev && (int)threadIdx.x < m) {
        const int k = threadIdx.x;
        const double lam = s_lam[k];
        double* y = Y + (size_t)k * L;
        double* tw = twb + (size_t)k * 4 * L;
        tri_inverse_iteration(sa, sb, m, lam, y, tw, tw + L, tw + 2 * L, tw + 3 * L, pivb + (size_t)k * L,
                              a.seed + 7919 * (uint64_t)k);
        a.evals[(size_t)c * nev + k] = lam;
        if (!(fabs(bt * y[m - 1]) <= a.tol * fmax(1.0, fabs(lam)))) atomicAnd(&s_done, 0);
      }
      __syncthreads();
      ortho_clustered(Y, L, m, ne, s_lam);
      __syncthreads();
      if (s_done || last) {
        converged = s_done;
        return true;
      }
    }
    return false;
  };
  for (;;) {
    // the steps up to the next check in a loop of their own: the check's
    // registers then displace the basis once per check, not in every step
    bool last;
    double bt;
    do {
      const int j = m;
      // v_j = w / beta; y = H v_j; alpha_j = Re <v_j, y>
      T v[R], y[R];
#pragma unroll
      for (int r = 0; r < R; ++r) set1(v[r], re1(w[r]) * sc, im1(w[r]) * sc);
      const double al = b.product(h, a.col, a.val, xs, sc, v, y);
      b.store(j, v);
      // the three-term update first (the big cancellation is then done before
      // any Gram-Schmidt coefficient is formed), then full reorthogonalization
      // against v_0..v_j, a second pass when the first removed more than half of
      // |w|^2 (always with dgks off)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        w[r] = y[r];
        add_scaled(w[r], -al, v[r]);
        add_scaled(w[r], -bprev, vp[r]);
        vp[r] = v[r];
      }
      double p1, pw = 0.0;
      for (int it = 0;; ++it) {
        double before;
        b.pass(j + 1, w, &before);
        if (it == 0) pw = before;
        p = 0.0;
#pragma unroll
        for (int r = 0; r < R; ++r) p = add_re(p, w[r], w[r]);
        publish();
        p1 = b.row_sum(p, 1);
        if (it == 1 || (a.dgks && !(p1 < 0.5 * pw))) break;
      }
      bt = sqrt(p1);
      m = j + 1;
      last = m == mmax || bt <= 1e-13 * (fabs(al) + bprev + 1e-300);
      if (threadIdx.x == 0) {
        sa[j] = al;
        sb[j] = bt;
      }
      bprev = bt;
      sc = 1.0 / bt;
    } while (!last && !(m >= nev && m >= cstart && m % a.check_every == 0));
    __syncthreads();
    if (ritz_check(last, bt)) break;
  }
  // Ritz vectors x_k = sum_l y_k[l] v_l, normalized, stored complex
  double2* X = a.evecs + base * nev;
  const int kk = nev < m ? nev : m;
  for (int k = 0; k < kk; ++k) {
    __syncthreads();
    T x[R];
    b.combine(m, Y + (size_t)k * L, x);
    p = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) p = add_re(p, x[r], x[r]);
    const double nn = sqrt(b.row_sum(p, 1));
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (b.g == 0 && b.on[r]) X[(size_t)k * n + b.row[r]] = make_double2(re1(x[r]) / nn, im1(x[r]) / nn);
  }
  for (int k = kk; k < nev; ++k) {
    for (int i = threadIdx.x; i < n; i += BT) X[(size_t)k * n + i] = make_double2(0.0, 0.0);
    if (threadIdx.x == 0) a.evals[(size_t)c * nev + k] = NAN;
  }
  if (threadIdx.x == 0) {
    a.steps[c] = m;
    a.conv[c] = converged;
  }
}

// bytes of LDS a workgroup needs before the LDS-held vectors
template <int NQ, int G, int R, class T>
size_t eigen_reg_fixed(int64_t nmax, int L, int nev) {
  using Basis = RegBasis<NQ, G, R, T>;
  const size_t ritz = 2 * (size_t)L + (size_t)nev * 5 * L + ((size_t)nev * L + 1) / 2;
  return 8 * ((ritz + 1) / 2 * 2 + ((size_t)nmax * Basis::D + 1) / 2 * 2 + Basis::fixed_doubles(L));
}

constexpr int kEigenLds = kRegLds - 2560;  // less the kernel's static arrays

template <int NQ, int G, int R, class T>
bool launch_eigen(EigenArgs a, unsigned nb, int n_cu, bool test, hipStream_t s) {
  using Basis = RegBasis<NQ, G, R, T>;
  const int L = std::min(a.max_steps, a.nmax);
  const size_t fixed = eigen_reg_fixed<NQ, G, R, T>(a.nmax, L, a.nev);
  if (test) return fixed <= (size_t)kEigenLds;
  static const hipError_t attr = hipFuncSetAttribute((const void*)eigen_reg_kernel<NQ, G, R, T>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, kEigenLds);
  HIP_CHECK(attr);
  a.lstride = L;
  // a workgroup's share of the CU's LDS, as in the Lanczos launch
  const int per_cu = std::max(1, (int)std::min<int64_t>(8 / (NQ * G), ((int64_t)nb + n_cu - 1) / n_cu));
  const size_t share = (size_t)kRegLds / per_cu / 1280 * 1280 - (kRegLds - kEigenLds);
  const size_t vec = (size_t)a.nmax * sizeof(T) * G;
  const int want = std::max(0, (L + G - 1) / G - Basis::S);
  const int cap = a.kl;  // eigen_lds_vectors
  a.kl = want > 0 && share > fixed ? (int)std::min<size_t>(want, (share - fixed) / vec) : 0;
  if (cap >= 0) a.kl = std::min(a.kl, cap);
  if (a.kl < want) a.kl = a.kl / Basis::B * Basis::B;  // whole batches where vectors follow in memory
  hipLaunchKernelGGL((eigen_reg_kernel<NQ, G, R, T>), dim3(nb), dim3(64 * NQ * G), fixed + vec * a.kl, s, a);
  HIP_CHECK(hipGetLastError());
  return true;
}

// The launch for a.nmax rows (test: whether its arrays fit the LDS), groups of
// waves per chain up to `groups`.
template <class T>
bool launch_eigen_type(const EigenArgs& a, unsigned nb, int n_cu, int groups, bool test, hipStream_t s) {
  switch (lanczos_reg_class(a.nmax)) {
    case 0:
      return groups >= 4   ? launch_eigen<1, 4, 1, T>(a, nb, n_cu, test, s)
             : groups == 2 ? launch_eigen<1, 2, 1, T>(a, nb, n_cu, test, s)
                           : launch_eigen<1, 1, 1, T>(a, nb, n_cu, test, s);
    case 1:
      return groups >= 4 ? launch_eigen<2, 4, 1, T>(a, nb, n_cu, test, s)
                         : launch_eigen<2, 2, 1, T>(a, nb, n_cu, test, s);
    case 2:
      return launch_eigen<3, 2, 1, T>(a, nb, n_cu, test, s);
    case 3:
      return launch_eigen<4, 2, 1, T>(a, nb, n_cu, test, s);
    case 4:
      return launch_eigen<4, 2, 2, T>(a, nb, n_cu, test, s);
    case 5:
      return launch_eigen<4, 2, 3, T>(a, nb, n_cu, test, s);
    default:
      return launch_eigen<4, 2, 4, T>(a, nb, n_cu, test, s);
  }
}

}  // namespace

}  // namespace imped
