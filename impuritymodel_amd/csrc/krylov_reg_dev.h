// Device code of the register-resident Krylov basis (krylov_reg.h).
#pragma once

#include <type_traits>

#include "krylov_reg.h"

namespace imped {

template <class T>
constexpr bool reg_real_v = sizeof(T) == sizeof(double);

__device__ __forceinline__ double re1(double x) { return x; }
__device__ __forceinline__ double re1(double2 x) { return x.x; }
__device__ __forceinline__ double im1(double) { return 0.0; }
__device__ __forceinline__ double im1(double2 x) { return x.y; }
__device__ __forceinline__ void set1(double& t, double r, double) { t = r; }
__device__ __forceinline__ void set1(double2& t, double r, double i) { t = make_double2(r, i); }

// Sums of products, every one an explicit fma in a fixed order, so that the bits do
// not depend on what the compiler contracts in an instance, and a real vector has the
// bits it has as a complex one with zero imaginary parts (or, times i, zero real
// parts): the terms with those parts are +-0.
// s + Re conj(a) b
__device__ __forceinline__ double add_re(double s, double a, double b) { return fma(a, b, s); }
__device__ __forceinline__ double add_re(double s, double2 a, double2 b) { return fma(a.y, b.y, fma(a.x, b.x, s)); }
// s + a b
__device__ __forceinline__ void add_mul(double& s, double a, double b) { s = fma(a, b, s); }
__device__ __forceinline__ void add_mul(double2& s, double2 a, double2 b) {
  s.x = fma(-a.y, b.y, fma(a.x, b.x, s.x));
  s.y = fma(a.y, b.x, fma(a.x, b.y, s.y));
}
// s + c a, real c
__device__ __forceinline__ void add_scaled(double& s, double c, double a) { s = fma(c, a, s); }
__device__ __forceinline__ void add_scaled(double2& s, double c, double2 a) {
  s.x = fma(c, a.x, s.x);
  s.y = fma(c, a.y, s.y);
}
__device__ __forceinline__ double sum1(double a, double b) { return a + b; }
__device__ __forceinline__ double2 sum1(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }

// f(integral_constant<int, 0>), ..., f(integral_constant<int, N - 1>): every
// index of a register array is then a constant, so the array stays in
// registers.
template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, I + 1>(f);
  }
}

// a and b of every lane exchanged so that their sum holds, in the lanes with
// bit 5 (W = 32) or bit 4 (W = 16) clear, a summed over the lane pair, in the
// others b.
template <int W>
__device__ __forceinline__ double halve_swap(double a, double b) {
  const unsigned al = (unsigned)__double2loint(a), ah = (unsigned)__double2hiint(a);
  const unsigned bl = (unsigned)__double2loint(b), bh = (unsigned)__double2hiint(b);
  if constexpr (W == 32) {
    const auto lo = __builtin_amdgcn_permlane32_swap(al, bl, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(ah, bh, false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
  } else {
    const auto lo = __builtin_amdgcn_permlane16_swap(al, bl, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
  }
}

// Eight values summed over the wave at once: lane l returns the sum of value
// l >> 3 (the eight lanes of a value hold the same number).
__device__ __forceinline__ double wave_sum8(const double (&x)[8], bool odd8) {
  double y[4], z[2];
#pragma unroll
  for (int k = 0; k < 4; ++k) y[k] = halve_swap<32>(x[k], x[k + 4]);
#pragma unroll
  for (int k = 0; k < 2; ++k) z[k] = halve_swap<16>(y[k], y[k + 2]);
  // lanes 8..15 of each row keep z[1]: send the other, receive from lane ^ 8
  const double send = odd8 ? z[0] : z[1];
  double r = (odd8 ? z[1] : z[0]) + dpp_move<0x128, 0xF>(send);  // row_ror:8
  r += dpp_move<0x141, 0xF>(r);                                  // row_half_mirror
  r += dpp_move<0x4E, 0xF>(r);                                   // quad_perm [2,3,0,1]
  r += dpp_move<0xB1, 0xF>(r);                                   // quad_perm [1,0,3,2]
  return r;
}

// Every value summed over the wave, by the same tree of lanes for N = 1 and 2.
template <int N>
__device__ __forceinline__ void wave_sums(double (&x)[N]) {
  double r = halve_swap<32>(x[0], x[N - 1]);  // value k in half k of the wave (N = 2)
  r = halve_swap<16>(r, r);
  r += dpp_move<0x128, 0xF>(r);  // row_ror:8
  r += dpp_move<0x141, 0xF>(r);  // row_half_mirror
  r += dpp_move<0x4E, 0xF>(r);   // quad_perm [2,3,0,1]
  r += dpp_move<0xB1, 0xF>(r);   // quad_perm [1,0,3,2]
#pragma unroll
  for (int k = 0; k < N; ++k)
    x[k] = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(r), 64 / N * k),
                            __builtin_amdgcn_readlane(__double2loint(r), 64 / N * k));
}

// Vectors of the basis in registers and entries of each row of H beside them:
// the most that the 256 registers of a thread hold without spilling (one wave alone
// also keeps all parts of the sums).
template <int W, int R, class T>
constexpr int reg_slots() {
  if (reg_real_v<T>) return R == 1 ? (W == 1 ? 56 : 72) : R == 2 ? 24 : 8;
  return R == 1 ? 32 : R == 2 ? 8 : 4;
}
template <int R, class T>
constexpr int reg_row_entries() {
  return R == 1 ? 8 : R == 2 || (reg_real_v<T> && R == 3) ? 4 : 0;
}

// One chain's basis and the Gram-Schmidt pass over it.
template <int NQ, int G, int R, class T>
struct RegBasis {
  static constexpr int W = NQ * G;                  // waves
  static constexpr int S = reg_slots<W, R, T>();    // register slots per thread
  static constexpr int B = reg_real_v<T> ? 8 : 4;   // vectors per reduction of eight values
  static constexpr int D = reg_real_v<T> ? 1 : 2;   // doubles per element
  static constexpr int F = kRegParts / G;           // parts of every sum that a group forms
  static_assert(G > 1 || W == 1, "one group of several waves: product has no case for it");
  static_assert(S % kRegParts == 0 && B % kRegParts == 0, "a part's vectors must not depend on where they sit");

  double vr[S][R], vi[reg_real_v<T> ? 1 : S][R];  // the register slots
  int lane, wave, q, g;
  bool odd8;
  int n, kl;  // kl: a multiple of B, or every vector past the registers
  int row[R];  // this thread's rows; past the chain's end: its last row, whose
  bool on[R];  // products are dropped (w is 0 there)
  T* vl;        // LDS: vector S*G + x at vl + x*n
  T* vg;        // memory: vector l at vg + l*n
  double* dotp;  // LDS [NQ][lcap * D * G]: dots of wave q's rows, by group and local index
  double* cw;    // LDS [W][lcap * D]: this wave's coefficients
  T* upd;       // LDS [G][NQ*64*R]: the groups' updates, and parts of H v (G > 1)
  double* red;  // LDS [2][W] and [kRegRowParts][NQ]
  int lcap;     // local vectors per group, a multiple of B

  static constexpr int kRed = 2 * W + kRegRowParts * NQ;  // (even)

  // doubles of LDS before the vectors for chains of K steps
  static __host__ __device__ int lcap_for(int K) { return ((K + G - 1) / G + B - 1) / B * B; }
  static __host__ __device__ size_t fixed_doubles(int K) {
    const size_t lc = (size_t)lcap_for(K) * D;
    return (size_t)NQ * G * lc + (NQ > 1 ? (size_t)W * lc : 0) + (G > 1 ? (size_t)G * NQ * 64 * R * D : 0) + kRed;
  }

  __device__ __forceinline__ void init(int n_, int K, int kl_, double* lds, T* vstore) {
    lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    q = wave % NQ;
    g = wave / NQ;
    odd8 = (lane & 8) != 0;
    n = n_;
    kl = kl_;
    lcap = lcap_for(K);
    dotp = lds;
    cw = NQ > 1 ? dotp + (size_t)NQ * G * lcap * D + (size_t)wave * lcap * D : dotp + (size_t)wave * lcap * D;
    double* p = dotp + (size_t)NQ * G * lcap * D + (NQ > 1 ? (size_t)W * lcap * D : 0);
    upd = reinterpret_cast<T*>(p);
    p += G > 1 ? (size_t)G * NQ * 64 * R * D : 0;
    red = p;
    p += kRed;
    vl = reinterpret_cast<T*>(p);
    vg = vstore;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      row[r] = (r * NQ + q) * 64 + lane;
      on[r] = row[r] < n;
      row[r] = on[r] ? row[r] : n - 1;
    }
    static_for<S * R>([&](auto k) __attribute__((always_inline)) {
      vr[k / R][k % R] = 0.0;
      if constexpr (!reg_real_v<T>) vi[k / R][k % R] = 0.0;
    });
  }

  template <int s, int r>
  __device__ __forceinline__ T slot() const {
    T t;
    if constexpr (reg_real_v<T>)
      t = vr[s][r];
    else
      t = make_double2(vr[s][r], vi[s][r]);
    return t;
  }

  // x becomes basis vector j
  __device__ __forceinline__ void store(int j, const T (&x)[R]) {
    if (j % G != g) return;
    const int li = __builtin_amdgcn_readfirstlane(j / G);
    if (li < S) {
      double xr[R], xi[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        xr[r] = re1(x[r]);
        xi[r] = im1(x[r]);
      }
      static_for<S / B>([&](auto b) __attribute__((always_inline)) {
        if (li / B == b) {
          static_for<B * R>([&](auto k) __attribute__((always_inline)) {
            constexpr int s = b * B + k / R, r = k % R;
            vr[s][r] = li == s ? xr[r] : vr[s][r];
            if constexpr (!reg_real_v<T>) vi[s][r] = li == s ? xi[r] : vi[s][r];
          });
          // no instruction: keeps the blocks of different b apart (merged,
          // they would address the array by a pointer)
          asm volatile("" ::"n"(b.value));
        }
      });
    } else if (li < S + kl) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (on[r]) vl[(size_t)((li - S) * G + g) * n + row[r]] = x[r];
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (on[r]) vg[(size_t)j * n + row[r]] = x[r];
    }
  }

  // local vectors [li, li + B) past the registers; entries past the count
  // (nl) repeat its last vector, their coefficients are 0
  __device__ __forceinline__ void fetch_lds(int li, int nl, T (&x)[B][R]) const {
#pragma unroll
    for (int s = 0; s < B; ++s) {
      const int k = li + s < nl ? li + s : nl - 1;
#pragma unroll
      for (int r = 0; r < R; ++r) x[s][r] = vl[(size_t)((k - S) * G + g) * n + row[r]];
    }
  }
  __device__ __forceinline__ void fetch_mem(int li, int nl, T (&x)[B][R]) const {
#pragma unroll
    for (int s = 0; s < B; ++s) {
      const int k = li + s < nl ? li + s : nl - 1;
#pragma unroll
      for (int r = 0; r < R; ++r) x[s][r] = vg[(size_t)(k * G + g) * n + row[r]];
    }
  }

  // dots of B vectors with w over this wave's rows, into the dots array
  template <class X>
  __device__ __forceinline__ void dot_batch(int li, int nl, const T (&w)[R], X&& x) {
    double p[8];
    static_for<B>([&](auto s) __attribute__((always_inline)) {
      double px = 0.0, py = 0.0;
      static_for<R>([&](auto r) __attribute__((always_inline)) {
        const T a = x(s, r);
        px = add_re(px, a, w[r]);
        if constexpr (!reg_real_v<T>) py = fma(-im1(a), re1(w[r]), fma(re1(a), im1(w[r]), py));
      });
      p[s * D] = px;
      if constexpr (!reg_real_v<T>) p[s * D + 1] = py;
    });
    double d = wave_sum8(p, odd8);
    if (li + (lane >> 3) / D >= nl) d = 0.0;
    double* dst = NQ > 1 ? dotp + ((size_t)q * G + g) * lcap * D : cw;
    if ((lane & 7) == 0) dst[(size_t)li * D + (lane >> 3)] = d;
  }

  template <class X>
  __device__ __forceinline__ void upd_batch(int li, T (&u)[F][R], X&& x) {
    const T* c = reinterpret_cast<const T*>(cw) + li;
    static_for<B>([&](auto s) __attribute__((always_inline)) {
      const T cs = c[s];
      static_for<R>([&](auto r) __attribute__((always_inline)) { add_mul(u[s % F][r], x(s, r), cs); });
    });
  }

  // The parts of one group, and of the groups, added up: (p0 + p2) + (p1 + p3)
  // whatever the number of groups (group g has parts g, g + G, ...).
  template <class U>
  static __device__ __forceinline__ U own_parts(const U (&p)[F]) {
    if constexpr (F == 4)
      return sum1(sum1(p[0], p[2]), sum1(p[1], p[3]));
    else if constexpr (F == 2)
      return sum1(p[0], p[1]);
    else
      return p[0];
  }
  __device__ __forceinline__ void put_part(int r, const T& t) const {
    upd[((size_t)g * R + r) * NQ * 64 + q * 64 + lane] = t;
  }
  __device__ __forceinline__ T get_part(int k, int r) const {
    return upd[((size_t)k * R + r) * NQ * 64 + q * 64 + lane];
  }
  __device__ __forceinline__ T all_parts(int r) const {
    if constexpr (G == 4)
      return sum1(sum1(get_part(0, r), get_part(2, r)), sum1(get_part(1, r), get_part(3, r)));
    else
      return sum1(get_part(0, r), get_part(1, r));
  }

  // sum of x over the chain's rows (x: this thread's part; the same in every
  // group), slot k of red (0: pass): one barrier
  __device__ __forceinline__ double row_sum(double x, int k) {
    x = wave_sum(x);
    if constexpr (W == 1) return x;
    if constexpr (NQ == 1) {
      __syncthreads();
      return x;
    }
    if (lane == 0) red[k * W + wave] = x;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int p = 0; p < NQ; ++p) t += red[k * W + g * NQ + p];
    return t;
  }

  // y = sc H x from RegRows (x in LDS), and Re <v, y>.  One barrier: the groups'
  // parts of y and each wave's parts of the product go to LDS together.
  template <class H>
  __device__ __forceinline__ double product(const H& h, const int32_t* col, const double2* val, const T* x, double sc,
                                            const T (&v)[R], T (&y)[R]) {
    double p[H::F];
#pragma unroll
    for (int f = 0; f < H::F; ++f) p[f] = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      T part[H::F];
      h.apply(r, col, val, x, part);
#pragma unroll
      for (int f = 0; f < H::F; ++f) {
        set1(part[f], re1(part[f]) * sc, im1(part[f]) * sc);
        p[f] = add_re(p[f], v[r], part[f]);
      }
      y[r] = part[0];
      if constexpr (H::F == 2) y[r] = sum1(part[0], part[1]);
    }
    wave_sums(p);
    if constexpr (W == 1) return p[0] + p[1];
    double* rp = red + 2 * W;
    if (g < kRegRowParts) {
      if (lane == 0) rp[g * NQ + q] = p[0];
#pragma unroll
      for (int r = 0; r < R; ++r) put_part(r, y[r]);
    }
    __syncthreads();
    double t[kRegRowParts];
#pragma unroll
    for (int k = 0; k < kRegRowParts; ++k) {
      t[k] = rp[k * NQ];
#pragma unroll
      for (int i = 1; i < NQ; ++i) t[k] += rp[k * NQ + i];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) y[r] = sum1(get_part(0, r), get_part(1, r));
    return t[0] + t[1];
  }

  // One classical Gram-Schmidt pass of w against vectors 0..m-1; *pw receives
  // |w|^2 before the pass.
  __device__ __forceinline__ void pass(int m, T (&w)[R], double* pw) {
    const int nl = __builtin_amdgcn_readfirstlane((m - g + G - 1) / G);  // this group's vectors
    double p = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) p = add_re(p, w[r], w[r]);
    p = wave_sum(p);
    if constexpr (NQ > 1) {
      if (lane == 0) red[wave] = p;
    }
    static_for<S / B>([&](auto bc) __attribute__((always_inline)) {
      constexpr int b = bc * B;
      if (b < nl) dot_batch(b, nl, w, [&](auto s, auto r) __attribute__((always_inline)) { return slot<b + s, r>(); });
    });
    const int n1 = nl < S + kl ? nl : S + kl;
    for (int li = S; li < n1; li += B) {
      T x[B][R];
      fetch_lds(li, n1, x);
      dot_batch(li, n1, w, [&](auto s, auto r) __attribute__((always_inline)) { return x[s][r]; });
    }
    for (int li = S + kl; li < nl; li += B) {
      T x[B][R];
      fetch_mem(li, nl, x);
      dot_batch(li, nl, w, [&](auto s, auto r) __attribute__((always_inline)) { return x[s][r]; });
    }
    __syncthreads();
    if constexpr (NQ > 1) {
      double t = 0.0;
#pragma unroll
      for (int k = 0; k < NQ; ++k) t += red[g * NQ + k];
      p = t;
      // this wave's copy of its group's coefficients
      // (whole batches: the entries past the count are 0)
      for (int x = lane; x < (nl + B - 1) / B * B * D; x += 64) {
        double c = dotp[(size_t)g * lcap * D + x];
#pragma unroll
        for (int k = 1; k < NQ; ++k) c += dotp[((size_t)k * G + g) * lcap * D + x];
        cw[x] = c;
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    *pw = p;
    T u[F][R];
#pragma unroll
    for (int k = 0; k < F * R; ++k) set1(u[k / R][k % R], 0.0, 0.0);
    static_for<S / B>([&](auto bc) __attribute__((always_inline)) {
      constexpr int b = bc * B;
      if (b < nl) upd_batch(b, u, [&](auto s, auto r) __attribute__((always_inline)) { return slot<b + s, r>(); });
    });
    for (int li = S; li < n1; li += B) {
      T x[B][R];
      fetch_lds(li, n1, x);
      upd_batch(li, u, [&](auto s, auto r) __attribute__((always_inline)) { return x[s][r]; });
    }
    for (int li = S + kl; li < nl; li += B) {
      T x[B][R];
      fetch_mem(li, nl, x);
      upd_batch(li, u, [&](auto s, auto r) __attribute__((always_inline)) { return x[s][r]; });
    }
    T d[R];
#pragma unroll
    for (int r = 0; r < R; ++r) d[r] = gather(u, r);
    if constexpr (G > 1) {
#pragma unroll
      for (int r = 0; r < R; ++r) put_part(r, d[r]);
      __syncthreads();
#pragma unroll
      for (int r = 0; r < R; ++r) d[r] = all_parts(r);
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (on[r]) set1(w[r], re1(w[r]) - re1(d[r]), im1(w[r]) - im1(d[r]));
  }
  static __device__ __forceinline__ T gather(const T (&u)[F][R], int r) {
    T p[F];
#pragma unroll
    for (int f = 0; f < F; ++f) p[f] = u[f][r];
    return own_parts(p);
  }

  // x = sum over l < m of y[l] v_l (real y; the same sum in every group)
  __device__ __forceinline__ void combine(int m, const double* y, T (&out)[R]) {
    const int nl = __builtin_amdgcn_readfirstlane((m - g + G - 1) / G);
    T u[F][R];
#pragma unroll
    for (int k = 0; k < F * R; ++k) set1(u[k / R][k % R], 0.0, 0.0);
    static_for<S>([&](auto s) __attribute__((always_inline)) {
      if (s < nl)
        static_for<R>([&](auto r) __attribute__((always_inline)) {
          add_scaled(u[s % F][r], y[s * G + g], slot<s, r>());
        });
    });
    const int n1 = nl < S + kl ? nl : S + kl;
    for (int li = S; li < n1; li += F)
#pragma unroll
      for (int f = 0; f < F; ++f)
        if (li + f < n1)
#pragma unroll
          for (int r = 0; r < R; ++r)
            add_scaled(u[f][r], y[(li + f) * G + g], vl[(size_t)((li + f - S) * G + g) * n + row[r]]);
#pragma unroll 4 / F
    for (int li = S + kl; li < nl; li += F)
#pragma unroll
      for (int f = 0; f < F; ++f)
        if (li + f < nl)
#pragma unroll
          for (int r = 0; r < R; ++r)
            add_scaled(u[f][r], y[(li + f) * G + g], vg[(size_t)((li + f) * G + g) * n + row[r]]);
    T d[R];
#pragma unroll
    for (int r = 0; r < R; ++r) d[r] = gather(u, r);
    if constexpr (G > 1) {
#pragma unroll
      for (int r = 0; r < R; ++r) put_part(r, d[r]);
      __syncthreads();
#pragma unroll
      for (int r = 0; r < R; ++r) d[r] = all_parts(r);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) set1(out[r], on[r] ? re1(d[r]) : 0.0, on[r] ? im1(d[r]) : 0.0);
  }
};

// The rows of H of one thread: entry e of a row counts to part e % kRegRowParts of its
// sum (the parts meet in RegBasis::product).  Group g takes part g % kRegRowParts, a
// single group both; up to HR of its entries are in registers, the rest read from
// memory.  (Four parts would divide the rows over four groups, but one group alone
// then spills: 18432 complex chains of 60 rows 2.7 ms, with two parts 2.5 ms; two
// chains of 100 rows in four groups each 406 and 403 us.)
template <int W, int G, int R, class T>
struct RegRows {
  static constexpr int HR = reg_row_entries<R, T>();
  static constexpr int N = G < kRegRowParts ? G : kRegRowParts;  // groups that share a row
  static constexpr int F = kRegRowParts / N;                     // parts that each forms
  static_assert(HR % 2 == 0, "an entry's part must not depend on where it sits");
  T h[R][HR ? HR : 1];
  int c[R][HR ? HR : 1];
  int cnt_wave[R];
  int64_t rest[R], end[R];

  __device__ __forceinline__ void load(const int64_t* rowptr, const int32_t* col, const double2* val, int g,
                                       const int (&row)[R], const bool (&on)[R]) {
    g %= N;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      int cnt = 0;
      rest[r] = end[r] = 0;
      int64_t e0 = 0;
      if (on[r]) {
        e0 = rowptr[row[r]] + g;
        end[r] = rowptr[row[r] + 1];
        const int64_t mine = end[r] > e0 ? (end[r] - e0 + N - 1) / N : 0;
        cnt = (int)(mine < HR ? mine : HR);
        rest[r] = e0 + (int64_t)cnt * N;
      }
#pragma unroll
      for (int k = 0; k < HR; ++k) {
        set1(h[r][k], 0.0, 0.0);
        c[r][k] = 0;
        if (k < cnt) {
          const double2 t = val[e0 + (int64_t)k * N];
          set1(h[r][k], t.x, t.y);
          c[r][k] = col[e0 + (int64_t)k * N];
        }
      }
      cnt_wave[r] = wave_max_int(cnt);
    }
  }

  // this group's parts of row r of H x (x in LDS)
  __device__ __forceinline__ void apply(int r, const int32_t* col, const double2* val, const T* x,
                                        T (&part)[F]) const {
#pragma unroll
    for (int f = 0; f < F; ++f) set1(part[f], 0.0, 0.0);
#pragma unroll
    for (int k0 = 0; k0 < HR; k0 += 4)
      if (k0 < cnt_wave[r]) {
        T t[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) t[u] = x[c[r][k0 + u]];
#pragma unroll
        for (int u = 0; u < 4; ++u) add_mul(part[u % F], h[r][k0 + u], t[u]);
      }
    // four entries per round trip (indices past the row clamped, their products skipped)
    for (int64_t e = rest[r]; e < end[r]; e += 4 * N) {
      T hh[4], t[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t k = e + u * N < end[r] ? e + u * N : end[r] - 1;
        const double2 z = val[k];
        set1(hh[u], z.x, z.y);
        t[u] = x[col[k]];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (e + u * N < end[r]) add_mul(part[u % F], hh[u], t[u]);
    }
  }
};

}  // namespace imped
