// lanczos_reg_kernel and its launch for one element type (krylov_reg.h);
// lanczos_reg_real.hip and lanczos_reg_cplx.hip instantiate it.
#pragma once

#include <algorithm>

#include "krylov_reg_dev.h"

namespace imped {

namespace {

// Fully reorthogonalized Lanczos of one chain per workgroup, the basis in
// registers (krylov_reg.h): the recurrence, the Gram-Schmidt rule and the
// outcome of lanczos_kernel with reorth = 1.  T = double: chains whose H and
// start vector (up to the factor i) are real, in real arithmetic.
//
// What bounds it: a chain's steps are a dependent sequence (two sums over the
// rows, the dots, the update), and inside a step the FP64 vector instructions
// of the two basis passes; with the basis on the chip no memory traffic is left.
// Before, chains beyond 80 KiB of basis kept it in memory (one wave per chain,
// HBM bound: 3.5 TB/s) and smaller ones in LDS (two chains per CU).  Measured
// on one MI355X, launch time before -> now: 1728 complex chains of 105..225
// rows, 150 steps, 29.7 -> 6.0 ms; 60 real chains of up to 733 rows, 150
// steps, 28.1 -> 2.0 ms; 18432 complex chains of 60 rows, 60 steps, 6.6 -> 2.5 ms;
// 873 of them 0.38 -> 0.19 ms.
template <int NQ, int G, int R, class T>
__global__ __launch_bounds__(64 * NQ * G, 2) void lanczos_reg_kernel(LanczosArgs a) {
  extern __shared__ double2 lds[];
  using Basis = RegBasis<NQ, G, R, T>;
  const int c = a.chain_list[blockIdx.x];
  const int n = (int)a.chain_n[c];
  const int64_t base = a.row_base[c];
  const int pure = a.pure ? a.pure[c] : 0;
  if (reg_real_v<T> != (pure != 0)) return;  // the launch of the other element type has it
  double* alpha = a.alpha + (size_t)c * a.K;
  double* beta = a.beta + (size_t)c * a.K;
  if (n == 0) {
    if (threadIdx.x == 0) {
      a.kout[c] = 0;
      a.status[c] = IMPED_OK;
    }
    return;
  }
  const int K = a.K < n ? a.K : n;
  T* xs = reinterpret_cast<T*>(lds);  // the residual, where the SpMV gathers from
  Basis b;
  b.init(n, K, a.kl, reinterpret_cast<double*>(lds) + ((size_t)a.nmax * Basis::D + 1) / 2 * 2,
         reinterpret_cast<T*>(a.vstore + (size_t)a.K * base));
  RegRows<NQ * G, G, R, T> h;
  h.load(a.rowptr + base, a.col, a.val, b.g, b.row, b.on);
  T w[R], vp[R];  // the residual; the latest basis vector
#pragma unroll
  for (int r = 0; r < R; ++r) {
    set1(w[r], 0.0, 0.0);
    if (b.on[r]) {
      const double2 t = a.v0[base + b.row[r]];
      if constexpr (reg_real_v<T>)
        w[r] = pure == 1 ? t.x : t.y;
      else
        w[r] = t;
    }
    set1(vp[r], 0.0, 0.0);
  }
  auto publish = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (b.g == 0 && b.on[r]) xs[b.row[r]] = w[r];
  };
  publish();
  __syncthreads();
  double sc = 1.0, beta_j = 0.0;
  int kdone = K, status = IMPED_OK;
  for (int j = 0;; ++j) {
    // v_j = w / beta; y = H v_j; alpha_j = Re <v_j, y>
    T v[R], y[R];
#pragma unroll
    for (int r = 0; r < R; ++r) set1(v[r], re1(w[r]) * sc, im1(w[r]) * sc);
    const double al = b.product(h, a.col, a.val, xs, sc, v, y);
    if (threadIdx.x == 0) alpha[j] = al;
    if (j + 1 == K) break;
    b.store(j, v);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      w[r] = y[r];
      add_scaled(w[r], -al, v[r]);
      add_scaled(w[r], -beta_j, vp[r]);
      vp[r] = v[r];
    }
    // full reorthogonalization against v_0..v_j; a second pass when the
    // first removed more than half of |w|^2
    double p, p1, pw = 0.0;
    for (int it = 0;; ++it) {
      double before;
      b.pass(j + 1, w, &before);
      if (it == 0) pw = before;
      p = 0.0;
#pragma unroll
      for (int r = 0; r < R; ++r) p = add_re(p, w[r], w[r]);
      publish();
      p1 = b.row_sum(p, 1);
      if (it == 1 || !(p1 < 0.5 * pw)) break;
    }
    beta_j = sqrt(p1);
    if (threadIdx.x == 0) beta[j] = beta_j;
    if (beta_j == 0.0) {
      status = IMPED_ERR_BREAKDOWN;
      kdone = j + 1;
      break;
    }
    sc = 1.0 / beta_j;
  }
  if (threadIdx.x == 0) {
    a.kout[c] = kdone;
    a.status[c] = status;
  }
}

// doubles of LDS a workgroup needs before the LDS-held vectors
template <int NQ, int G, int R, class T>
size_t lanczos_reg_fixed(int64_t nmax, int K) {
  using Basis = RegBasis<NQ, G, R, T>;
  return ((size_t)nmax * Basis::D + 1) / 2 * 2 + Basis::fixed_doubles(K);
}

template <int NQ, int G, int R, class T>
void launch_reg(LanczosArgs a, unsigned nb, int n_cu, hipStream_t s) {
  using Basis = RegBasis<NQ, G, R, T>;
  static const hipError_t attr =
      hipFuncSetAttribute((const void*)lanczos_reg_kernel<NQ, G, R, T>, hipFuncAttributeMaxDynamicSharedMemorySize,
                          kRegLds);
  HIP_CHECK(attr);
  const int K = std::min(a.K, a.nmax);
  const size_t fixed = lanczos_reg_fixed<NQ, G, R, T>(a.nmax, K) * 8;
  // a workgroup's share of the CU's LDS: as many workgroups as the launch
  // gives a CU, at most the two waves per SIMD that the registers allow
  const int per_cu = std::max(1, (int)std::min<int64_t>(8 / (NQ * G), ((int64_t)nb + n_cu - 1) / n_cu));
  const size_t share = (size_t)kRegLds / per_cu / 1280 * 1280;
  const size_t vec = (size_t)a.nmax * sizeof(T) * G;
  const int want = std::max(0, (K - 1 + G - 1) / G - Basis::S);  // the last vector is never read
  // want = 0 covers launches of empty chains only (vec = 0)
  a.kl = want > 0 && share > fixed ? (int)std::min<size_t>(want, (share - fixed) / vec) : 0;
  if (a.kl < want) a.kl = a.kl / Basis::B * Basis::B;  // whole batches where vectors follow in memory
  const size_t bytes = fixed + vec * a.kl;
  if (bytes > (size_t)kRegLds) throw HipError{"lanczos: coefficients exceed the LDS"};
  hipLaunchKernelGGL((lanczos_reg_kernel<NQ, G, R, T>), dim3(nb), dim3(64 * NQ * G), bytes, s, a);
  HIP_CHECK(hipGetLastError());
}

// The launch for a.nmax rows, groups of waves per chain up to `groups`.
template <class T>
void launch_reg_type(const LanczosArgs& a, unsigned nb, int n_cu, int groups, hipStream_t s) {
  switch (lanczos_reg_class(a.nmax)) {
    case 0:
      if (groups >= 4)
        launch_reg<1, 4, 1, T>(a, nb, n_cu, s);
      else if (groups == 2)
        launch_reg<1, 2, 1, T>(a, nb, n_cu, s);
      else
        launch_reg<1, 1, 1, T>(a, nb, n_cu, s);
      break;
    case 1:
      if (groups >= 4)
        launch_reg<2, 4, 1, T>(a, nb, n_cu, s);
      else
        launch_reg<2, 2, 1, T>(a, nb, n_cu, s);
      break;
    case 2:
      launch_reg<3, 2, 1, T>(a, nb, n_cu, s);
      break;
    case 3:
      launch_reg<4, 2, 1, T>(a, nb, n_cu, s);
      break;
    case 4:
      launch_reg<4, 2, 2, T>(a, nb, n_cu, s);
      break;
    case 5:
      launch_reg<4, 2, 3, T>(a, nb, n_cu, s);
      break;
    default:
      launch_reg<4, 2, 4, T>(a, nb, n_cu, s);
  }
}

}  // namespace

}  // namespace imped
