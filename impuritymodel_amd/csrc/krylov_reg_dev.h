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

// Vectors of the basis in registers and entries of each row of H beside them:
// the most that the 256 registers of a thread hold without spilling.
template <int W, int R, class T>
constexpr int reg_slots() {
  if (reg_real_v<T>) return R == 1 ? 72 : R == 2 ? 24 : 8;
  return R == 1 ? (W == 1 ? 36 : 32) : R == 2 ? 8 : 4;
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
  double* red;  // LDS [3][W]
  int lcap;     // local vectors per group, a multiple of B

  // doubles of LDS before the vectors for chains of K steps
  static __host__ __device__ int lcap_for(int K) { return ((K + G - 1) / G + B - 1) / B * B; }
  static __host__ __device__ size_t fixed_doubles(int K) {
    const size_t lc = (size_t)lcap_for(K) * D;
    return (size_t)NQ * G * lc + (NQ > 1 ? (size_t)W * lc : 0) + (G > 1 ? (size_t)G * NQ * 64 * R * D : 0) + 3 * W + (W & 1);
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
    p += 3 * W + (W & 1);
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
  template <class F>
  __device__ __forceinline__ void dot_batch(int li, int nl, const T (&w)[R], F&& x) {
    double p[8];
    static_for<B>([&](auto s) __attribute__((always_inline)) {
      double px = 0.0, py = 0.0;
      static_for<R>([&](auto r) __attribute__((always_inline)) {
        const T a = x(s, r);
        px += re1(a) * re1(w[r]);
        if constexpr (!reg_real_v<T>) {
          px += im1(a) * im1(w[r]);
          py += re1(a) * im1(w[r]);
          py -= im1(a) * re1(w[r]);
        }
      });
      p[s * D] = px;
      if constexpr (!reg_real_v<T>) p[s * D + 1] = py;
    });
    double d = wave_sum8(p, odd8);
    if (li + (lane >> 3) / D >= nl) d = 0.0;
    double* dst = NQ > 1 ? dotp + ((size_t)q * G + g) * lcap * D : cw;
    if ((lane & 7) == 0) dst[(size_t)li * D + (lane >> 3)] = d;
  }

  template <class F>
  __device__ __forceinline__ void upd_batch(int li, T (&u0)[R], T (&u1)[R], F&& x) {
    const T* c = reinterpret_cast<const T*>(cw) + li;
    static_for<B>([&](auto s) __attribute__((always_inline)) {
      const T cs = c[s];
      static_for<R>([&](auto r) __attribute__((always_inline)) {
        const T a = x(s, r);
        T& u = s & 1 ? u1[r] : u0[r];
        if constexpr (reg_real_v<T>) {
          u += a * cs;
        } else {
          u.x += a.x * cs.x;
          u.x -= a.y * cs.y;
          u.y += a.x * cs.y;
          u.y += a.y * cs.x;
        }
      });
    });
  }

  // sum of x over the chain's rows (x: this thread's part; the same in every
  // group), slot k of three used in turn: one barrier
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

  // (yr, yi) <- the groups' parts of H v summed; returns Re <v, H v>.  One
  // barrier: the parts and each wave's share of the product go to LDS together.
  __device__ __forceinline__ double product(const T (&v)[R], double (&yr)[R], double (&yi)[R]) {
    double p = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) p += re1(v[r]) * yr[r] + im1(v[r]) * yi[r];
    if constexpr (G == 1) return row_sum(p, 2);
    p = wave_sum(p);
    if (lane == 0) red[2 * W + wave] = p;
#pragma unroll
    for (int r = 0; r < R; ++r) set1(upd[((size_t)g * R + r) * NQ * 64 + q * 64 + lane], yr[r], yi[r]);
    __syncthreads();
    p = 0.0;
#pragma unroll
    for (int k = 0; k < W; ++k) p += red[2 * W + k];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      yr[r] = yi[r] = 0.0;
#pragma unroll
      for (int k = 0; k < G; ++k) {
        const T t = upd[((size_t)k * R + r) * NQ * 64 + q * 64 + lane];
        yr[r] += re1(t);
        yi[r] += im1(t);
      }
    }
    return p;
  }

  // One classical Gram-Schmidt pass of w against vectors 0..m-1; *pw receives
  // |w|^2 before the pass.
  __device__ __forceinline__ void pass(int m, T (&w)[R], double* pw) {
    const int nl = __builtin_amdgcn_readfirstlane((m - g + G - 1) / G);  // this group's vectors
    double p = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) p += re1(w[r]) * re1(w[r]) + im1(w[r]) * im1(w[r]);
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
    T u0[R], u1[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      set1(u0[r], 0.0, 0.0);
      set1(u1[r], 0.0, 0.0);
    }
    static_for<S / B>([&](auto bc) __attribute__((always_inline)) {
      constexpr int b = bc * B;
      if (b < nl) upd_batch(b, u0, u1, [&](auto s, auto r) __attribute__((always_inline)) { return slot<b + s, r>(); });
    });
    for (int li = S; li < n1; li += B) {
      T x[B][R];
      fetch_lds(li, n1, x);
      upd_batch(li, u0, u1, [&](auto s, auto r) __attribute__((always_inline)) { return x[s][r]; });
    }
    for (int li = S + kl; li < nl; li += B) {
      T x[B][R];
      fetch_mem(li, nl, x);
      upd_batch(li, u0, u1, [&](auto s, auto r) __attribute__((always_inline)) { return x[s][r]; });
    }
    if constexpr (G == 1) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (on[r]) set1(w[r], re1(w[r]) - (re1(u0[r]) + re1(u1[r])), im1(w[r]) - (im1(u0[r]) + im1(u1[r])));
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r)
        set1(upd[((size_t)g * R + r) * NQ * 64 + q * 64 + lane], re1(u0[r]) + re1(u1[r]), im1(u0[r]) + im1(u1[r]));
      __syncthreads();
#pragma unroll
      for (int r = 0; r < R; ++r) {
        double ux = 0.0, uy = 0.0;
#pragma unroll
        for (int k = 0; k < G; ++k) {
          const T t = upd[((size_t)k * R + r) * NQ * 64 + q * 64 + lane];
          ux += re1(t);
          uy += im1(t);
        }
        if (on[r]) set1(w[r], re1(w[r]) - ux, im1(w[r]) - uy);
      }
    }
  }

  // x = sum over l < m of y[l] v_l (real y; the same sum in every group)
  __device__ __forceinline__ void combine(int m, const double* y, T (&out)[R]) {
    const int nl = __builtin_amdgcn_readfirstlane((m - g + G - 1) / G);
    double ur[R], ui[R];
#pragma unroll
    for (int r = 0; r < R; ++r) ur[r] = ui[r] = 0.0;
    auto add = [&](double c, int r, const T& t) __attribute__((always_inline)) {
      ur[r] += c * re1(t);
      if constexpr (!reg_real_v<T>) ui[r] += c * im1(t);
    };
    static_for<S>([&](auto s) __attribute__((always_inline)) {
      if (s < nl)
        static_for<R>([&](auto r) __attribute__((always_inline)) { add(y[s * G + g], r, slot<s, r>()); });
    });
    const int n1 = nl < S + kl ? nl : S + kl;
    for (int li = S; li < n1; ++li)
#pragma unroll
      for (int r = 0; r < R; ++r) add(y[li * G + g], r, vl[(size_t)((li - S) * G + g) * n + row[r]]);
#pragma unroll 4
    for (int li = S + kl; li < nl; ++li)
#pragma unroll
      for (int r = 0; r < R; ++r) add(y[li * G + g], r, vg[(size_t)(li * G + g) * n + row[r]]);
    if constexpr (G > 1) {
#pragma unroll
      for (int r = 0; r < R; ++r) set1(upd[((size_t)g * R + r) * NQ * 64 + q * 64 + lane], ur[r], ui[r]);
      __syncthreads();
#pragma unroll
      for (int r = 0; r < R; ++r) {
        ur[r] = ui[r] = 0.0;
#pragma unroll
        for (int k = 0; k < G; ++k) {
          const T t = upd[((size_t)k * R + r) * NQ * 64 + q * 64 + lane];
          ur[r] += re1(t);
          ui[r] += im1(t);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) set1(out[r], on[r] ? ur[r] : 0.0, on[r] ? ui[r] : 0.0);
  }
};

// The rows of H of one thread: group g takes entries g, g + G, ... of each row,
// up to HR of them in registers, the rest read from memory (the groups'
// products of a row meet in RegBasis::product).
template <int W, int G, int R, class T>
struct RegRows {
  static constexpr int HR = reg_row_entries<R, T>();
  T h[R][HR ? HR : 1];
  int c[R][HR ? HR : 1];
  int cnt_wave[R];
  int64_t rest[R], end[R];

  __device__ __forceinline__ void load(const int64_t* rowptr, const int32_t* col, const double2* val, int g,
                                       const int (&row)[R], const bool (&on)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      int cnt = 0;
      rest[r] = end[r] = 0;
      int64_t e0 = 0;
      if (on[r]) {
        e0 = rowptr[row[r]] + g;
        end[r] = rowptr[row[r] + 1];
        const int64_t mine = end[r] > e0 ? (end[r] - e0 + G - 1) / G : 0;
        cnt = (int)(mine < HR ? mine : HR);
        rest[r] = e0 + (int64_t)cnt * G;
      }
#pragma unroll
      for (int k = 0; k < HR; ++k) {
        set1(h[r][k], 0.0, 0.0);
        c[r][k] = 0;
        if (k < cnt) {
          const double2 t = val[e0 + (int64_t)k * G];
          set1(h[r][k], t.x, t.y);
          c[r][k] = col[e0 + (int64_t)k * G];
        }
      }
      cnt_wave[r] = wave_max_int(cnt);
    }
  }

  // this group's part of row r of H x (x in LDS)
  __device__ __forceinline__ void apply(int r, const int32_t* col, const double2* val, const T* x, double* yr,
                                        double* yi) const {
    double ax = 0.0, ay = 0.0, bx = 0.0, by = 0.0;
    auto add = [](double& sx, double& sy, const T& a, const T& b) {
      sx += re1(a) * re1(b);
      if constexpr (!reg_real_v<T>) {
        sx -= im1(a) * im1(b);
        sy += re1(a) * im1(b);
        sy += im1(a) * re1(b);
      }
    };
#pragma unroll
    for (int k0 = 0; k0 < HR; k0 += 4)
      if (k0 < cnt_wave[r]) {
        T t[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) t[u] = x[c[r][k0 + u]];
        add(ax, ay, h[r][k0], t[0]);
        add(bx, by, h[r][k0 + 1], t[1]);
        add(ax, ay, h[r][k0 + 2], t[2]);
        add(bx, by, h[r][k0 + 3], t[3]);
      }
    // four entries per round trip (indices past the row clamped, their products skipped)
    for (int64_t e = rest[r]; e < end[r]; e += 4 * G) {
      T hh[4], t[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t k = e + u * G < end[r] ? e + u * G : end[r] - 1;
        const double2 z = val[k];
        set1(hh[u], z.x, z.y);
        t[u] = x[col[k]];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (e + u * G < end[r]) add(ax, ay, hh[u], t[u]);
    }
    *yr = ax + bx;
    *yi = ay + by;
  }
};

}  // namespace imped
