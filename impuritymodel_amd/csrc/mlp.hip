// Surrogate network kernels: an ensemble of E fully connected GELU networks
// of identical shape, trained and evaluated together (blockIdx.z = member).
//
// * gemm_nt_kernel: every GEMM, C[m][n] = sum_k A[m][k] B[n][k] with both
//   operands k-contiguous and padded to whole tiles: forward (X W^T), input
//   gradient (dZ W, from a transposed copy of W) and weight gradient (dZ^T X,
//   from transposed copies that the producing epilogues write).  Epilogues fuse the bias, GELU (pre-activation kept in FP32 for the
//   backward pass), the loss and its gradient, the GELU derivative, the bias
//   gradients and the Adam update.
// * gather_kernel, loss_sum_kernel: minibatch inputs and the losses.
//
// BF16 copies of weights and activations are stored with rows padded to a
// multiple of 64 entries, the padding zero, so no load is bounds-checked.  The
// epilogues write those zeros whatever the sum is: an infinite activation times
// a padding row of weights is NaN, and one NaN in the padding of a row would
// reach every output of its sample (or, from a padding sample, every weight).
#include <cmath>
#include <cstring>
#include <memory>

#include "common.h"
#include "mlp.h"

namespace imped {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// round-to-nearest-even float -> bfloat16 (NaN stays NaN)
__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

// GELU(x) = x Phi(x) and its derivative Phi(x) + x phi(x), Phi(x) = (1 +
// erf(x / sqrt 2)) / 2 (training: full-precision erf)
__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float x) {
  const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
  const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
  return cdf + x * pdf;
}

// erf by the rational approximation of Abramowitz and Stegun, Handbook of
// Mathematical Functions, eq. 7.1.26 (after Hastings): erf(x) = 1 - (a1 t +
// a2 t^2 + a3 t^3 + a4 t^4 + a5 t^5) exp(-x^2), t = 1 / (1 + p x) for x >= 0,
// odd in x, absolute error at most 1.5e-7 (5.3e-7 in FP32 arithmetic) -- far
// below the BF16 rounding (2^-8 relative) of the activations it feeds, at a
// fraction of the instructions of the full-precision erf.  Inference only
// (the epilogue of a hidden layer evaluates sixteen per lane); training keeps
// gelu above, so a trained network does not depend on it.
__device__ __forceinline__ float erf_as(float x) {
  const float ax = fabsf(x);
  const float t = __builtin_amdgcn_rcpf(1.0f + 0.3275911f * ax);
  const float poly =
      t * (0.254829592f + t * (-0.284496736f + t * (1.421413741f + t * (-1.453152027f + t * 1.061405429f))));
  return copysignf(1.0f - poly * __expf(-ax * ax), x);
}
__device__ __forceinline__ float gelu_inference(float x) {
  return 0.5f * x * (1.0f + erf_as(x * 0.70710678118654752f));
}

constexpr int TM = 64, TN = 64;

enum { NT_GELU, NT_MSE, NT_DGELU, NT_GRAD, NT_ADAM, NT_HIDDEN, NT_OUT };

// gemm_nt_kernel: M, N rows of A and B that hold data, out of mp, np (multiples
// of 64; rows between are zero or meet zeros), K a multiple of 64.
struct NtArgs {
  const uint16_t* A;
  int64_t lda, a_z;
  const uint16_t* B;
  int64_t ldb, b_z;
  int M, N, mp, np, K;
  const float* bias;  // forward: [N] per member
  int64_t bias_z;
  const float* Af;  // with AF: A in FP32 [M][lda] (shared by the members), entries past lda taken as 0
  float* out;       // NT_OUT: result [M][N] per member
  float* z;      // NT_GELU: pre-activations written, NT_DGELU: read; [mp][np]
  uint16_t* C;   // NT_GELU, NT_MSE, NT_DGELU, NT_HIDDEN: BF16 result [mp][np]
  uint16_t* CT;  //   (but NT_HIDDEN) and transposed [np][mp]; both per member mp * np
  // NT_MSE: targets (row idx[m], or m without idx) and the sum of squares of each tile
  const float* T;
  const int32_t* idx;
  double* lossp;
  // NT_GRAD, NT_ADAM: gradient or parameters of the layer, flat [M][N], then the biases [M]
  float *g, *w, *m, *v;
  int64_t p_z, b_off;
  uint16_t *wb, *wbT;  // NT_ADAM: BF16 copies [mp][np] and [np][mp]
  int64_t wb_z;
  float lr, b1, b2, eps, bc1, bc2;
};

// Eight FP32 values rounded to BF16, packed as the BF16 row chunk.
__device__ __forceinline__ uint4 pack_bf16x8(const float4& a, const float4& b) {
  uint4 r;
  r.x = (uint32_t)f2bf(a.x) | ((uint32_t)f2bf(a.y) << 16);
  r.y = (uint32_t)f2bf(a.z) | ((uint32_t)f2bf(a.w) << 16);
  r.z = (uint32_t)f2bf(b.x) | ((uint32_t)f2bf(b.y) << 16);
  r.w = (uint32_t)f2bf(b.z) | ((uint32_t)f2bf(b.w) << 16);
  return r;
}

// Adam step of one parameter from its gradient; returns the new value.
__device__ __forceinline__ float adam_step(const NtArgs& a, int64_t o, float g) {
  const float mi = a.b1 * a.m[o] + (1.0f - a.b1) * g;
  const float vi = a.b2 * a.v[o] + (1.0f - a.b2) * g * g;
  a.m[o] = mi;
  a.v[o] = vi;
  const float w = a.w[o] - a.lr * (mi / a.bc1) / (sqrtf(vi / a.bc2) + a.eps);
  a.w[o] = w;
  return w;
}

// blockIdx -> (member, column tile, row tile) for the eight XCDs, which take the
// workgroups round-robin in launch order (x fastest) and each have their own L2:
// with the launch order, XCD i got output-column tile i of every row tile and
// member, so each XCD fetched every activation tile (eight fetches per tile).
// Renumbered so that each XCD takes one contiguous run of tiles, ordered
// member, column tile, row tile (rows fastest): an XCD's run covers whole
// columns of one or two members, every weight tile is fetched by one XCD and
// every activation tile by about two.  Same arithmetic per tile.
__device__ __forceinline__ void xcd_tile(int& z, int& bx, int& by) {
  z = blockIdx.z, bx = blockIdx.x, by = blockIdx.y;
  const int gx = gridDim.x, gy = gridDim.y, tiles = gx * gy * gridDim.z;
  if ((tiles & 7) == 0) {
    const int l = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
    const int q = (l & 7) * (tiles >> 3) + (l >> 3);  // a bijection of [0, tiles) when 8 | tiles
    z = q / (gx * gy);
    const int r = q - z * gx * gy;
    bx = r / gy;
    by = r - bx * gy;
  }
}

// One 64 x 64 tile per workgroup of four waves (a 32 x 32 accumulator each), K
// in steps of 64 through two LDS buffers: the next step's 16-byte loads are in
// flight while this step's four MFMAs per wave run, one barrier a step.
//
// What bounds it: at these sizes a launch is a few dependent load latencies
// plus the epilogue's stores; small tiles, because 1024 x 512 outputs of five
// members are only 640 of them.  Measured, five members of 8-512-512-512-1000
// on one MI355X: a 512 x 512 layer at 256 rows 9.9 -> 8.3 us a launch, at 1001
// rows 18.6 -> 11.2 us (both against K staged 256 deep, bounds-checked); a
// training step of 1024 rows 1.63 -> 0.24 ms, of which the separate bias
// gradients (one thread per column, 220 us a layer), the loss (an FP64 atomic
// per 256 values, 242 us) and transposing loads were 1.3 ms.
template <int EPI, bool AF = false>
__global__ __launch_bounds__(256) void gemm_nt_kernel(NtArgs g) {
  constexpr int SK = 64, LK = SK + 8;  // rows of 144 bytes spread over the banks
  __shared__ __align__(16) uint16_t As[2][TM][LK], Bs[2][TN][LK];
  __shared__ double red[4];
  int z, bx, by;
  xcd_tile(z, bx, by);
  const int m0 = by * TM, n0 = bx * TN;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const int sr = t >> 2, sc = (t & 3) * 16;  // this thread's staged row and its 16 entries
  const uint16_t* pa = AF ? nullptr : g.A + (int64_t)z * g.a_z + (int64_t)(m0 + sr) * g.lda + sc;
  // AF: rows past M read the last one (their outputs are dropped)
  const float* paf = AF ? g.Af + (int64_t)(m0 + sr < g.M ? m0 + sr : g.M - 1) * g.lda + sc : nullptr;
  const auto load_a = [&](int k, uint4& lo, uint4& hi) {
    if constexpr (AF) {
      lo = hi = make_uint4(0, 0, 0, 0);
      if (sc + k < g.lda)
        lo = pack_bf16x8(*reinterpret_cast<const float4*>(paf + k), *reinterpret_cast<const float4*>(paf + k + 4));
      if (sc + k + 8 < g.lda)
        hi = pack_bf16x8(*reinterpret_cast<const float4*>(paf + k + 8), *reinterpret_cast<const float4*>(paf + k + 12));
    } else {
      lo = *reinterpret_cast<const uint4*>(pa + k);
      hi = *reinterpret_cast<const uint4*>(pa + k + 8);
    }
  };
  const uint16_t* pb = g.B + (int64_t)z * g.b_z + (int64_t)(n0 + sr) * g.ldb + sc;
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  constexpr bool weights = EPI == NT_GRAD || EPI == NT_ADAM;
  const bool row_sums = weights && bx == 0;  // the bias gradients: sums of A's rows
  float rs = 0.0f;
  uint4 a0, a1;
  load_a(0, a0, a1);
  uint4 b0 = *reinterpret_cast<const uint4*>(pb), b1 = *reinterpret_cast<const uint4*>(pb + 8);
  for (int k0 = 0, buf = 0; k0 < g.K; k0 += SK, buf ^= 1) {
    *reinterpret_cast<uint4*>(&As[buf][sr][sc]) = a0;
    *reinterpret_cast<uint4*>(&As[buf][sr][sc + 8]) = a1;
    *reinterpret_cast<uint4*>(&Bs[buf][sr][sc]) = b0;
    *reinterpret_cast<uint4*>(&Bs[buf][sr][sc + 8]) = b1;
    if (row_sums) {
      const uint32_t u[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
#pragma unroll
      for (int i = 0; i < 8; ++i) rs += __uint_as_float(u[i] << 16) + __uint_as_float(u[i] & 0xffff0000u);
    }
    __syncthreads();
    if (k0 + SK < g.K) {
      load_a(k0 + SK, a0, a1);
      b0 = *reinterpret_cast<const uint4*>(pb + k0 + SK);
      b1 = *reinterpret_cast<const uint4*>(pb + k0 + SK + 8);
    }
#pragma unroll
    for (int kk = 0; kk < SK; kk += 16) {
      // lane l supplies row l%32 and k = kk + 8*(l/32) .. +7 of each operand
      const int kq = kk + 8 * (lane >> 5);
      const uint4 a = *reinterpret_cast<const uint4*>(&As[buf][wm + (lane & 31)][kq]);
      const uint4 b = *reinterpret_cast<const uint4*>(&Bs[buf][wn + (lane & 31)][kq]);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc,
                                                    0, 0, 0);
    }
  }
  // accumulator r of lane l holds row 8*(r/4) + 4*(l/32) + r%4, column l%32
  const int n = n0 + wn + (lane & 31), mb = m0 + wm + 4 * (lane >> 5);
  if constexpr (weights) {
    if (row_sums) {  // the four threads of a row
      rs += __shfl_xor(rs, 1);
      rs += __shfl_xor(rs, 2);
      if ((t & 3) == 0 && m0 + sr < g.M) {
        const int64_t o = (int64_t)z * g.p_z + g.b_off + m0 + sr;
        if constexpr (EPI == NT_GRAD)
          g.g[o] = rs;
        else
          adam_step(g, o, rs);
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint16_t h[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = mb + 8 * q + r;
        const int64_t o = (int64_t)z * g.p_z + (int64_t)m * g.N + n;
        h[r] = 0;
        if (m < g.M && n < g.N) {
          if constexpr (EPI == NT_GRAD) {
            g.g[o] = acc[4 * q + r];
          } else {
            h[r] = f2bf(adam_step(g, o, acc[4 * q + r]));
            g.wb[(int64_t)z * g.wb_z + (int64_t)m * g.np + n] = h[r];
          }
        }
      }
      if constexpr (EPI == NT_ADAM)
        *reinterpret_cast<uint2*>(g.wbT + (int64_t)z * g.wb_z + (int64_t)n * g.mp + mb + 8 * q) =
            make_uint2(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16);
    }
  } else if constexpr (EPI == NT_OUT || EPI == NT_HIDDEN) {
    // the column's bias read once and added to every accumulator before the
    // first store: first used inside the per-row branches, it would put a wait
    // for every earlier store between the stores
    const float bn = n < g.N ? g.bias[(int64_t)z * g.bias_z + n] : 0.0f;
    const uint16_t col = n < g.N ? 0xffff : 0;  // a mask, not a branch around the GELU
    float v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      v[r] = acc[r] + bn;
      asm volatile("" : "+v"(v[r]));  // no instruction: keeps the sum here
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = mb + 8 * (r >> 2) + (r & 3);
      if constexpr (EPI == NT_HIDDEN)
        g.C[((int64_t)z * g.mp + m) * g.np + n] = f2bf(gelu_inference(v[r])) & col;
      else if (m < g.M && n < g.N)
        g.out[((int64_t)z * g.M + m) * g.N + n] = v[r];
    }
  } else {
    const int64_t cz = (int64_t)z * g.mp * g.np;
    float bn = 0.0f;
    if constexpr (EPI != NT_DGELU) bn = n < g.N ? g.bias[(int64_t)z * g.bias_z + n] : 0.0f;
    double sq = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint16_t h[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = mb + 8 * q + r;
        const int64_t o = cz + (int64_t)m * g.np + n;
        const float v = acc[4 * q + r] + bn;
        const bool data = m < g.M && n < g.N;
        h[r] = 0;
        if constexpr (EPI == NT_GELU) {
          g.z[o] = v;
          h[r] = data ? f2bf(gelu(v)) : (uint16_t)0;
        } else if constexpr (EPI == NT_DGELU) {
          h[r] = data ? f2bf(v * gelu_grad(g.z[o])) : (uint16_t)0;
        } else {
          if (data) {
            const float d = v - g.T[(int64_t)(g.idx ? g.idx[m] : m) * g.N + n];
            h[r] = f2bf(2.0f * d / (float)((int64_t)g.M * g.N));
            sq += (double)d * (double)d;
          }
        }
        g.C[o] = h[r];
      }
      *reinterpret_cast<uint2*>(g.CT + cz + (int64_t)n * g.mp + mb + 8 * q) =
          make_uint2(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16);
    }
    if constexpr (EPI == NT_MSE) {
      sq = wave_sum(sq);
      if (lane == 0) red[wave] = sq;
      __syncthreads();
      if (t == 0) g.lossp[((int64_t)z * gridDim.y + by) * gridDim.x + bx] = red[0] + red[1] + red[2] + red[3];
    }
  }
}

// out[i] = sum of part[i*tiles ..] / count, one wave per value
__global__ __launch_bounds__(64) void loss_sum_kernel(const double* part, int tiles, double count, double* out) {
  double s = 0.0;
  for (int k = threadIdx.x; k < tiles; k += 64) s += part[(int64_t)blockIdx.x * tiles + k];
  s = wave_sum(s);
  if (threadIdx.x == 0) out[blockIdx.x] = s / count;
}

// x [B][d] in BF16 with rows padded to ld entries (the padding stays zero)
__global__ void to_bf16_kernel(const float* x, int64_t n, int d, int ld, uint16_t* y) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i / d * ld + i % d] = f2bf(x[i]);
}

// BF16 copies of one layer's weights W [out][in] of every member: wb [op][ip]
// and its transpose wbT [ip][op], zero-padded (members w_z and wb_z apart)
__global__ void pack_weights_kernel(const float* w, int64_t w_z, int out, int in, int op, int ip, uint16_t* wb,
                                    uint16_t* wbT, int64_t wb_z) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)op * ip) return;
  const int64_t z = blockIdx.y;
  const int o = (int)(i / ip), k = (int)(i % ip);
  wb[z * wb_z + i] = o < out && k < in ? f2bf(w[z * w_z + (int64_t)o * in + k]) : (uint16_t)0;
  const int kt = (int)(i / op), ot = (int)(i % op);
  wbT[z * wb_z + i] = ot < out && kt < in ? f2bf(w[z * w_z + (int64_t)ot * in + kt]) : (uint16_t)0;
}

// minibatch inputs (row idx[b] of X, or b without idx) in BF16, xb [bp][ld]
// and xT [ld][bp]; rows from B on are zero
__global__ void gather_kernel(const float* X, int dx, const int32_t* idx, int B, int bp, int ld, uint16_t* xb,
                              uint16_t* xT) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= bp) return;
  const int64_t r = b < B ? (idx ? idx[b] : b) : 0;
  for (int j = 0; j < dx; ++j) {
    const uint16_t h = b < B ? f2bf(X[r * dx + j]) : (uint16_t)0;
    xb[(int64_t)b * ld + j] = h;
    xT[(int64_t)j * bp + b] = h;
  }
}

// Sum over a 256-thread workgroup, broadcast to every thread.
__device__ __forceinline__ double sum256(double v, double* red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  __syncthreads();  // red may still be read by the previous call
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return red[0] + red[1] + red[2] + red[3];
}

// Ensemble statistics of one sample per workgroup, from the outputs
// y [E][B][D]: member spectra m_e = max(y_e / scale, 0) / area_e (area =
// sum_d w_d (.), the trapezoid rule when w holds its weights), their mean
// renormalized to unit area, the disagreement
// dis = (1/E) sum_e sum_d w_d |m_e,d - mean_d| and, when target is given,
// the misfit l1 = sum_d w_d |mean_d - target_d|.  E <= 64; the general
// path (ensemble_stats_reg_kernel covers E <= 8, D <= 1024).
__global__ __launch_bounds__(256) void ensemble_stats_kernel(const float* y, int E, int B, int D, const double* w,
                                                             double scale, const double* target, double* mean,
                                                             double* dis, double* l1) {
  __shared__ double red[4];
  __shared__ double area[64];
  const int b = blockIdx.x;
  for (int e = 0; e < E; ++e) {
    const float* ye = y + ((int64_t)e * B + b) * D;
    double p = 0.0;
    for (int d = threadIdx.x; d < D; d += 256) p += w[d] * fmax((double)ye[d] / scale, 0.0);
    p = sum256(p, red);
    if (threadIdx.x == 0) area[e] = p;
  }
  __syncthreads();
  double* mb = mean + (int64_t)b * D;
  double pm = 0.0;
  for (int d = threadIdx.x; d < D; d += 256) {
    double acc = 0.0;
    for (int e = 0; e < E; ++e) acc += fmax((double)y[((int64_t)e * B + b) * D + d] / scale, 0.0) / area[e];
    acc /= (double)E;
    mb[d] = acc;
    pm += w[d] * acc;
  }
  const double marea = sum256(pm, red);
  double pd = 0.0, pl = 0.0;
  for (int d = threadIdx.x; d < D; d += 256) {
    const double mn = mb[d] / marea;
    mb[d] = mn;
    for (int e = 0; e < E; ++e)
      pd += w[d] * fabs(fmax((double)y[((int64_t)e * B + b) * D + d] / scale, 0.0) / area[e] - mn);
    if (target) pl += w[d] * fabs(mn - target[d]);
  }
  pd = sum256(pd, red);
  if (target) pl = sum256(pl, red);
  if (threadIdx.x == 0) {
    dis[b] = pd / (double)E;
    if (target) l1[b] = pl;
  }
}

// Sums of NV values over a 256-thread workgroup, broadcast to every thread;
// red [4][NV] is this round's own LDS, so one barrier suffices.
template <int NV>
__device__ __forceinline__ void sums256(double (&v)[NV], double (*red)[NV]) {
#pragma unroll
  for (int i = 0; i < NV; ++i) v[i] = wave_sum(v[i]);
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int i = 0; i < NV; ++i) red[threadIdx.x >> 6][i] = v[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NV; ++i) v[i] = red[0][i] + red[1][i] + red[2][i] + red[3][i];
}

// The same statistics with the sample's member outputs loaded once into
// registers (EM members, D <= 256 K; thread t holds d = t + 256 k): each
// statistic is register arithmetic and one workgroup reduction (DPP wave
// sums, then LDS), three rounds in all, and every division is by a
// reciprocal formed once.
template <int K, int EM>
__global__ __launch_bounds__(256) void ensemble_stats_reg_kernel(const float* y, int E, int B, int D,
                                                                 const double* w, double scale,
                                                                 const double* target, double* mean, double* dis,
                                                                 double* l1) {
  __shared__ double red_a[4][EM], red_m[4][1], red_d[4][2];
  const int t = threadIdx.x;
  const int b = blockIdx.x;
  const double inv_scale = 1.0 / scale;
  double v[EM][K], wd[K];
#pragma unroll
  for (int e = 0; e < EM; ++e)
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int d = t + 256 * k;
      v[e][k] = (e < E && d < D) ? fmax((double)y[((int64_t)e * B + b) * D + d] * inv_scale, 0.0) : 0.0;
    }
  double tg[K];  // the target's values, loaded with the rest (mean may be NULL: not written)
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int d = t + 256 * k;
    wd[k] = d < D ? w[d] : 0.0;
    tg[k] = target && d < D ? target[d] : 0.0;
  }
  double inv_area[EM];
#pragma unroll
  for (int e = 0; e < EM; ++e) {
    double p = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) p += wd[k] * v[e][k];
    inv_area[e] = p;
  }
  sums256<EM>(inv_area, red_a);
#pragma unroll
  for (int e = 0; e < EM; ++e) inv_area[e] = e < E ? 1.0 / inv_area[e] : 0.0;
  double mn[K], pm[1] = {0.0};
  const double inv_e = 1.0 / (double)E;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    double acc = 0.0;
#pragma unroll
    for (int e = 0; e < EM; ++e) acc += v[e][k] * inv_area[e];
    mn[k] = acc * inv_e;
    pm[0] += wd[k] * mn[k];
  }
  sums256<1>(pm, red_m);
  const double inv_marea = 1.0 / pm[0];
  double pd[2] = {0.0, 0.0};
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int d = t + 256 * k;
    const double m = mn[k] * inv_marea;
    double s = 0.0;
#pragma unroll
    for (int e = 0; e < EM; ++e)
      if (e < E) s += fabs(v[e][k] * inv_area[e] - m);
    pd[0] += wd[k] * s;
    if (d < D) {
      if (mean) mean[(int64_t)b * D + d] = m;
      if (target) pd[1] += wd[k] * fabs(m - tg[k]);
    }
  }
  sums256<2>(pd, red_d);
  if (t == 0) {
    dis[b] = pd[0] * inv_e;
    if (target) l1[b] = pd[1];
  }
}

template <int EPI, bool AF = false>
void gemm_nt(const NtArgs& g, int E, hipStream_t s) {
  hipLaunchKernelGGL((gemm_nt_kernel<EPI, AF>), dim3(g.np / TN, g.mp / TM, E), dim3(256), 0, s, g);
  HIP_CHECK(hipGetLastError());
}

inline int pad64(int n) { return (n + 63) / 64 * 64; }

}  // namespace

// ------------------------------------------------------------------ network state

// Page-locked host memory mapped into the device's address space: kernels
// read small per-call inputs from it and write small results into it, so
// they move without a copy dispatch.  Every call that uses it synchronizes
// its stream before returning, so the next call may overwrite it.
struct HostIO {
  void* h = nullptr;  // host address
  void* d = nullptr;  // device address of the same memory
  size_t bytes = 0;
  void reserve(size_t n) {
    if (n <= bytes) return;
    release();
    HIP_CHECK(hipHostMalloc(&h, n, hipHostMallocDefault));
    HIP_CHECK(hipHostGetDevicePointer(&d, h, 0));
    bytes = n;
  }
  void release() {
    if (h) (void)hipHostFree(h);
    h = d = nullptr;
    bytes = 0;
  }
  HostIO() = default;
  HostIO(const HostIO&) = delete;
  HostIO& operator=(const HostIO&) = delete;
  ~HostIO() { release(); }
};

struct Mlp {
  int E = 0, L = 0, max_batch = 0;
  std::vector<int> dims;            // L + 1
  std::vector<int64_t> w_off, b_off;  // per layer offsets in a member's flat parameter vector
  int64_t P = 0;                    // parameters per member
  int64_t step = 0;                 // Adam steps taken
  std::vector<int> pd;              // widths padded to multiples of 64
  std::vector<int64_t> wbo;         // per layer offsets in a member's BF16 weights
  int64_t PB = 0;                   // BF16 weights per member
  DevBuf w, g, m, v;                // [E][P] fp32 master, gradient, Adam moments
  DevBuf wb, wbT;                   // [E][PB] bf16 weights: layer l [pd[l+1]][pd[l]], and transposed
  static constexpr int MAXL = 16;
  // per layer: activation bf16 [E][rows][pd[l+1]] (rows: the batch padded to a
  // multiple of 64); training: transposed, pre-activation fp32, dZ and transposed
  DevBuf hb[MAXL], hT[MAXL], zf[MAXL], dz[MAXL], dzT[MAXL];
  int act_rows = 0, train_rows = 0;
  DevBuf xb, xT, out, loss;         // minibatch input bf16 [rows][pd[0]], transposed; output fp32 [E][B][dL]; losses
  DevBuf dX, dY;                    // data set (fp32)
  DevBuf sw, smean, st;             // ensemble statistics: area weights, mean [B][dL], misfit target [dL]
  HostIO xin, sout;                 // batch input x [B][d0] (fp32); disagreement [B] and misfit [B]
  std::vector<double> sw_host, st_host;  // the area weights and target last uploaded
  // Prediction graphs (input conversion, forward GEMMs, statistics): one
  // launch instead of six, so the GPU does not wait for the host between
  // kernels.  Keyed by everything baked into the captured launches.
  struct PredictGraph {
    std::vector<uintptr_t> key;
    hipGraphExec_t exec = nullptr;
  };
  std::vector<PredictGraph> graphs;
  hipStream_t cap = nullptr;  // capture stream
  ~Mlp() {
    for (auto& g : graphs) (void)hipGraphExecDestroy(g.exec);
    if (cap) (void)hipStreamDestroy(cap);
  }
  int64_t n_data = 0;
};

namespace {

// A buffer of n bytes, all zero when it had to grow (the padding of BF16
// arrays is written by nobody, so it stays zero whatever the batch).
void reserve_zero(DevBuf& b, size_t n, hipStream_t s) {
  if (n <= b.bytes) return;
  b.reserve(n);
  HIP_CHECK(hipMemsetAsync(b.p, 0, b.bytes, s));
}

void alloc_acts(Mlp& net, int B, hipStream_t s) {
  const int rows = pad64(std::max(B, net.max_batch));
  if (rows <= net.act_rows) return;
  for (int l = 0; l + 1 < net.L; ++l) reserve_zero(net.hb[l], (size_t)net.E * rows * net.pd[l + 1] * 2, s);
  reserve_zero(net.xb, (size_t)rows * net.pd[0] * 2, s);
  net.out.reserve((size_t)net.E * rows * net.dims[net.L] * 4);
  net.act_rows = rows;
}

void alloc_train(Mlp& net, int B, hipStream_t s) {
  alloc_acts(net, B, s);
  const int rows = net.act_rows;
  if (rows <= net.train_rows) return;
  for (int l = 0; l < net.L; ++l) {
    const size_t n = (size_t)net.E * rows * net.pd[l + 1];
    if (l + 1 < net.L) {
      reserve_zero(net.hT[l], n * 2, s);
      net.zf[l].reserve(n * 4);
    }
    net.dz[l].reserve(n * 2);
    net.dzT[l].reserve(n * 2);
  }
  reserve_zero(net.xT, (size_t)rows * net.pd[0] * 2, s);
  net.train_rows = rows;
}

// Forward pass of a prediction: every member on B samples, outputs in out.
// x_f32: the first layer reads FP32 inputs there (else the BF16 copy in xb).
void forward(Mlp& net, int B, hipStream_t s, const float* x_f32 = nullptr) {
  const int rows = pad64(B);
  for (int l = 0; l < net.L; ++l) {
    NtArgs g{};
    g.A = l ? net.hb[l - 1].as<uint16_t>() : net.xb.as<uint16_t>();
    g.lda = g.K = net.pd[l];
    g.a_z = l ? (int64_t)rows * net.pd[l] : 0;
    g.B = net.wb.as<uint16_t>() + net.wbo[l];
    g.ldb = net.pd[l];
    g.b_z = net.PB;
    g.M = B;
    g.N = net.dims[l + 1];
    g.mp = rows;
    g.np = net.pd[l + 1];
    g.bias = net.w.as<float>() + net.b_off[l];
    g.bias_z = net.P;
    g.C = net.hb[l].as<uint16_t>();
    g.out = net.out.as<float>();
    const bool af = l == 0 && x_f32;
    if (af) {
      g.Af = x_f32;
      g.lda = net.dims[0];
    }
    TimedLaunch tl("mlp_gemm", s);
    if (l + 1 < net.L)
      af ? gemm_nt<NT_HIDDEN, true>(g, net.E, s) : gemm_nt<NT_HIDDEN>(g, net.E, s);
    else
      af ? gemm_nt<NT_OUT, true>(g, net.E, s) : gemm_nt<NT_OUT>(g, net.E, s);
  }
}

int loss_tiles(const Mlp& net, int B) { return net.pd[net.L] / TN * (pad64(B) / TM); }

// Adam's numbers of one step; null pointers elsewhere mean gradients only.
struct AdamStep {
  float lr, b1, b2, eps, bc1, bc2;
};

// One training pass of every member over the minibatch whose inputs are in
// xb/xT: forward, loss and its gradient against T (rows idx, or 0..B-1), then
// per layer, from the last, the input gradient and the weight gradient.  With
// adam the weight gradients go straight into the update (the layer's old
// weights were read by the input gradient queued before it), else to g.
// lossp: [E][loss_tiles] sums of squares.
void train_pass(Mlp& net, int B, const float* T, const int32_t* idx, double* lossp, const AdamStep* adam,
                hipStream_t s) {
  const int L = net.L, rows = pad64(B);
  for (int l = 0; l < L; ++l) {
    NtArgs g{};
    g.A = l ? net.hb[l - 1].as<uint16_t>() : net.xb.as<uint16_t>();
    g.lda = g.K = net.pd[l];
    g.a_z = l ? (int64_t)rows * net.pd[l] : 0;
    g.B = net.wb.as<uint16_t>() + net.wbo[l];
    g.ldb = net.pd[l];
    g.b_z = net.PB;
    g.M = B;
    g.N = net.dims[l + 1];
    g.mp = rows;
    g.np = net.pd[l + 1];
    g.bias = net.w.as<float>() + net.b_off[l];
    g.bias_z = net.P;
    TimedLaunch tl("mlp_gemm", s);
    if (l + 1 < L) {
      g.z = net.zf[l].as<float>();
      g.C = net.hb[l].as<uint16_t>();
      g.CT = net.hT[l].as<uint16_t>();
      gemm_nt<NT_GELU>(g, net.E, s);
    } else {
      g.C = net.dz[l].as<uint16_t>();
      g.CT = net.dzT[l].as<uint16_t>();
      g.T = T;
      g.idx = idx;
      g.lossp = lossp;
      gemm_nt<NT_MSE>(g, net.E, s);
    }
  }
  for (int l = L - 1; l >= 0; --l) {
    if (l > 0) {
      // dZ_{l-1}[b][i] = (sum_o dZ[b][o] W[o][i]) * gelu'(Z_{l-1}[b][i])
      NtArgs g{};
      g.A = net.dz[l].as<uint16_t>();
      g.lda = g.K = net.pd[l + 1];
      g.a_z = (int64_t)rows * net.pd[l + 1];
      g.B = net.wbT.as<uint16_t>() + net.wbo[l];
      g.ldb = net.pd[l + 1];
      g.b_z = net.PB;
      g.M = B;
      g.N = net.dims[l];
      g.mp = rows;
      g.np = net.pd[l];
      g.z = net.zf[l - 1].as<float>();
      g.C = net.dz[l - 1].as<uint16_t>();
      g.CT = net.dzT[l - 1].as<uint16_t>();
      TimedLaunch tl("mlp_gemm", s);
      gemm_nt<NT_DGELU>(g, net.E, s);
    }
    // dW[o][i] = sum_b dZ[b][o] X[b][i]
    NtArgs g{};
    g.A = net.dzT[l].as<uint16_t>();
    g.lda = g.ldb = g.K = rows;
    g.a_z = (int64_t)rows * net.pd[l + 1];
    g.B = l ? net.hT[l - 1].as<uint16_t>() : net.xT.as<uint16_t>();
    g.b_z = l ? (int64_t)rows * net.pd[l] : 0;
    g.M = net.dims[l + 1];
    g.N = net.dims[l];
    g.mp = net.pd[l + 1];
    g.np = net.pd[l];
    g.p_z = net.P;
    g.b_off = net.b_off[l] - net.w_off[l];
    if (adam) {
      g.w = net.w.as<float>() + net.w_off[l];
      g.m = net.m.as<float>() + net.w_off[l];
      g.v = net.v.as<float>() + net.w_off[l];
      g.wb = net.wb.as<uint16_t>() + net.wbo[l];
      g.wbT = net.wbT.as<uint16_t>() + net.wbo[l];
      g.wb_z = net.PB;
      g.lr = adam->lr;
      g.b1 = adam->b1;
      g.b2 = adam->b2;
      g.eps = adam->eps;
      g.bc1 = adam->bc1;
      g.bc2 = adam->bc2;
      TimedLaunch tl("mlp_adam", s);
      gemm_nt<NT_ADAM>(g, net.E, s);
    } else {
      g.g = net.g.as<float>() + net.w_off[l];
      TimedLaunch tl("mlp_gemm", s);
      gemm_nt<NT_GRAD>(g, net.E, s);
    }
  }
}

// Minibatch inputs of X (rows idx, or 0..B-1) into xb and xT.
void gather_batch(Mlp& net, const float* X, const int32_t* idx, int B, hipStream_t s) {
  const int rows = pad64(B);
  hipLaunchKernelGGL(gather_kernel, dim3(blocks_for(rows, 64)), dim3(64), 0, s, X, net.dims[0], idx, B, rows,
                     net.pd[0], net.xb.as<uint16_t>(), net.xT.as<uint16_t>());
  HIP_CHECK(hipGetLastError());
}

// x into the mapped input buffer; convert_batch_input launches the
// conversion, which reads it there (no copy dispatch).
void stage_batch_input(Mlp& net, const float* x_host, int B) {
  const int64_t n = (int64_t)B * net.dims[0];
  net.xin.reserve(n * sizeof(float));
  std::memcpy(net.xin.h, x_host, n * sizeof(float));
}

void convert_batch_input(Mlp& net, int B, hipStream_t s) {
  const int64_t n = (int64_t)B * net.dims[0];
  hipLaunchKernelGGL(to_bf16_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, static_cast<const float*>(net.xin.d),
                     n, net.dims[0], net.pd[0], net.xb.as<uint16_t>());
  HIP_CHECK(hipGetLastError());
}

void upload_batch_input(Mlp& net, const float* x_host, int B, hipStream_t s) {
  stage_batch_input(net, x_host, B);
  convert_batch_input(net, B, s);
}

}  // namespace

Mlp* mlp_create(int E, int L, const int32_t* dims, int max_batch) {
  auto net = std::make_unique<Mlp>();
  net->E = E;
  net->L = L;
  net->dims.assign(dims, dims + L + 1);
  int64_t off = 0;
  for (int l = 0; l < L; ++l) {
    net->w_off.push_back(off);
    off += (int64_t)dims[l + 1] * dims[l];
    net->b_off.push_back(off);
    off += dims[l + 1];
  }
  // members start 16-element aligned so every BF16 row load stays aligned
  net->P = (off + 15) / 16 * 16;
  for (int l = 0; l <= L; ++l) net->pd.push_back(pad64(dims[l]));
  for (int l = 0; l < L; ++l) {
    net->wbo.push_back(net->PB);
    net->PB += (int64_t)net->pd[l + 1] * net->pd[l];
  }
  const int64_t tot = (int64_t)E * net->P;
  net->w.reserve(tot * 4);
  net->wb.reserve((size_t)E * net->PB * 2);
  net->wbT.reserve((size_t)E * net->PB * 2);
  net->g.reserve(tot * 4);
  net->m.reserve(tot * 4);
  net->v.reserve(tot * 4);
  HIP_CHECK(hipMemset(net->w.p, 0, tot * 4));
  HIP_CHECK(hipMemset(net->wb.p, 0, (size_t)E * net->PB * 2));
  HIP_CHECK(hipMemset(net->wbT.p, 0, (size_t)E * net->PB * 2));
  HIP_CHECK(hipMemset(net->g.p, 0, tot * 4));
  HIP_CHECK(hipMemset(net->m.p, 0, tot * 4));
  HIP_CHECK(hipMemset(net->v.p, 0, tot * 4));
  net->max_batch = std::max(max_batch, 1);
  alloc_acts(*net, net->max_batch, nullptr);
  HIP_CHECK(hipStreamSynchronize(nullptr));
  return net.release();
}

void mlp_destroy(Mlp* net) { delete net; }
int64_t mlp_param_count(const Mlp& net) { return net.P; }
int64_t mlp_data_count(const Mlp& net) { return net.n_data; }
int mlp_layers(const Mlp& net, int32_t* dims) {
  if (dims)
    for (int l = 0; l <= net.L; ++l) dims[l] = net.dims[l];
  return net.L;
}

void mlp_get_params(Mlp& net, float* params, hipStream_t s) {
  d2h(params, net.w.p, (size_t)net.E * net.P, s);
  stream_sync(s);
}

void mlp_set_params(Mlp& net, const float* params, hipStream_t s) {
  const int64_t tot = (int64_t)net.E * net.P;
  HIP_CHECK(hipMemcpyAsync(net.w.p, params, tot * 4, hipMemcpyHostToDevice, s));
  for (int l = 0; l < net.L; ++l) {
    const int64_t n = (int64_t)net.pd[l + 1] * net.pd[l];
    hipLaunchKernelGGL(pack_weights_kernel, dim3(blocks_for(n, 256), net.E), dim3(256), 0, s,
                       net.w.as<float>() + net.w_off[l], net.P, net.dims[l + 1], net.dims[l], net.pd[l + 1], net.pd[l],
                       net.wb.as<uint16_t>() + net.wbo[l], net.wbT.as<uint16_t>() + net.wbo[l], net.PB);
    HIP_CHECK(hipGetLastError());
  }
  HIP_CHECK(hipMemsetAsync(net.m.p, 0, tot * 4, s));
  HIP_CHECK(hipMemsetAsync(net.v.p, 0, tot * 4, s));
  stream_sync(s);
  net.step = 0;
}

void mlp_forward(Mlp& net, const float* x_host, int B, float* y_host, hipStream_t s) {
  alloc_acts(net, B, s);
  upload_batch_input(net, x_host, B, s);
  forward(net, B, s);  // the network's outputs as predictions form them
  d2h(y_host, net.out.p, (size_t)net.E * B * net.dims[net.L], s);
  stream_sync(s);
}

namespace {

// Uploads a host vector of D doubles to dev when it differs from the copy
// last uploaded (the grid's weights and a fit's target stay the same from
// call to call).
void upload_on_change(DevBuf& dev, std::vector<double>& last, const double* host, int D, hipStream_t s) {
  if (last.size() != (size_t)D || std::memcmp(last.data(), host, D * sizeof(double)) != 0) {
    last.assign(host, host + D);
    h2d(dev, last.data(), D, s);
  }
}

}  // namespace

namespace {

template <int K>
bool launch_stats_reg_k(int E, int B, const float* y, int D, const double* w, double scale, const double* tgt,
                        double* m, double* dis, double* l1, hipStream_t s) {
  const dim3 g(B), t(256);
  switch (E) {
    case 1: hipLaunchKernelGGL((ensemble_stats_reg_kernel<K, 1>), g, t, 0, s, y, E, B, D, w, scale, tgt, m, dis, l1); break;
    case 2: hipLaunchKernelGGL((ensemble_stats_reg_kernel<K, 2>), g, t, 0, s, y, E, B, D, w, scale, tgt, m, dis, l1); break;
    case 3: hipLaunchKernelGGL((ensemble_stats_reg_kernel<K, 3>), g, t, 0, s, y, E, B, D, w, scale, tgt, m, dis, l1); break;
    case 4: hipLaunchKernelGGL((ensemble_stats_reg_kernel<K, 4>), g, t, 0, s, y, E, B, D, w, scale, tgt, m, dis, l1); break;
    case 5: hipLaunchKernelGGL((ensemble_stats_reg_kernel<K, 5>), g, t, 0, s, y, E, B, D, w, scale, tgt, m, dis, l1); break;
    case 6: hipLaunchKernelGGL((ensemble_stats_reg_kernel<K, 6>), g, t, 0, s, y, E, B, D, w, scale, tgt, m, dis, l1); break;
    case 7: hipLaunchKernelGGL((ensemble_stats_reg_kernel<K, 7>), g, t, 0, s, y, E, B, D, w, scale, tgt, m, dis, l1); break;
    case 8: hipLaunchKernelGGL((ensemble_stats_reg_kernel<K, 8>), g, t, 0, s, y, E, B, D, w, scale, tgt, m, dis, l1); break;
    default: return false;
  }
  return true;
}

// The register kernel for E <= 8 members and K values per thread; false if none fits.
bool launch_stats_reg(int K, int E, int B, const float* y, int D, const double* w, double scale, const double* tgt,
                      double* m, double* dis, double* l1, hipStream_t s) {
  if (K == 1) return launch_stats_reg_k<1>(E, B, y, D, w, scale, tgt, m, dis, l1, s);
  if (K == 2) return launch_stats_reg_k<2>(E, B, y, D, w, scale, tgt, m, dis, l1, s);
  return launch_stats_reg_k<4>(E, B, y, D, w, scale, tgt, m, dis, l1, s);
}

// Conversion, forward pass and ensemble statistics of B staged samples.
void enqueue_predict(Mlp& net, int B, double scale, bool with_target, bool with_mean, hipStream_t s) {
  if (net.dims[0] % 8 == 0) {
    forward(net, B, s, static_cast<const float*>(net.xin.d));  // inputs read from the mapped buffer
  } else {
    convert_batch_input(net, B, s);
    forward(net, B, s);
  }
  const int D = net.dims[net.L];
  const double* tgt = with_target ? net.st.as<double>() : nullptr;
  const float* y = net.out.as<float>();
  // disagreement and misfit are written straight into the mapped result buffer
  double *m = net.smean.as<double>(), *dis = static_cast<double*>(net.sout.d), *l1 = dis + B;
  const double* w = net.sw.as<double>();
  if (net.E <= 8 && D <= 1024 && !with_mean) m = nullptr;  // the register kernel writes no means then
  if (net.E > 8 || D > 1024 ||
      !launch_stats_reg(D <= 256 ? 1 : D <= 512 ? 2 : 4, net.E, B, y, D, w, scale, tgt, m, dis, l1, s))
    hipLaunchKernelGGL(ensemble_stats_kernel, dim3(B), dim3(256), 0, s, y, net.E, B, D, w, scale, tgt, m, dis, l1);
  HIP_CHECK(hipGetLastError());
}

// The captured enqueue_predict for this call's sizes and buffers.
hipGraphExec_t predict_graph(Mlp& net, int B, double scale, bool with_target, bool with_mean) {
  uint64_t sbits;
  std::memcpy(&sbits, &scale, sizeof(sbits));
  std::vector<uintptr_t> key = {(uintptr_t)B, (uintptr_t)sbits, (uintptr_t)with_target, (uintptr_t)with_mean,
                                (uintptr_t)net.xin.d, (uintptr_t)net.sout.d, (uintptr_t)net.smean.p,
                                (uintptr_t)net.sw.p, (uintptr_t)net.st.p, (uintptr_t)net.xb.p,
                                (uintptr_t)net.wb.p, (uintptr_t)net.w.p, (uintptr_t)net.out.p};
  for (int l = 0; l < net.L; ++l) key.push_back((uintptr_t)net.hb[l].p);
  for (const auto& g : net.graphs)
    if (g.key == key) return g.exec;
  if (!net.cap) HIP_CHECK(hipStreamCreateWithFlags(&net.cap, hipStreamNonBlocking));
  HIP_CHECK(hipStreamBeginCapture(net.cap, hipStreamCaptureModeThreadLocal));
  hipGraph_t graph = nullptr;
  try {
    enqueue_predict(net, B, scale, with_target, with_mean, net.cap);
  } catch (...) {
    (void)hipStreamEndCapture(net.cap, &graph);
    if (graph) (void)hipGraphDestroy(graph);
    throw;
  }
  HIP_CHECK(hipStreamEndCapture(net.cap, &graph));
  hipGraphExec_t exec = nullptr;
  const hipError_t ie = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  HIP_CHECK(ie);
  if (net.graphs.size() >= 8) {
    // every call synchronizes before returning: no launch of the oldest graph is in flight
    HIP_CHECK(hipGraphExecDestroy(net.graphs.front().exec));
    net.graphs.erase(net.graphs.begin());
  }
  net.graphs.push_back(Mlp::PredictGraph{key, exec});
  return exec;
}

}  // namespace

void mlp_predict(Mlp& net, const float* x_host, int B, const double* w_host, double scale, const double* target_host,
                 double* mean_host, double* dis_host, double* l1_host, hipStream_t s) {
  mlp_predict_begin(net, x_host, B, w_host, scale, target_host, mean_host, s);
  mlp_predict_end(net, B, target_host != nullptr, dis_host, l1_host, s);
}

void mlp_predict_begin(Mlp& net, const float* x_host, int B, const double* w_host, double scale,
                       const double* target_host, double* mean_host, hipStream_t s) {
  alloc_acts(net, B, s);
  stage_batch_input(net, x_host, B);
  const int D = net.dims[net.L];
  upload_on_change(net.sw, net.sw_host, w_host, D, s);
  if (target_host) upload_on_change(net.st, net.st_host, target_host, D, s);
  net.smean.reserve((size_t)B * D * sizeof(double));
  net.sout.reserve((size_t)2 * B * sizeof(double));
  // per-kernel timing needs direct launches
  const bool with_target = target_host != nullptr, with_mean = mean_host != nullptr;
  if (timing_enabled() || !g_tuning.mlp_graph)
    enqueue_predict(net, B, scale, with_target, with_mean, s);
  else
    HIP_CHECK(hipGraphLaunch(predict_graph(net, B, scale, with_target, with_mean), s));
  if (mean_host) d2h(mean_host, net.smean.p, (size_t)B * D, s);
}

void mlp_predict_end(Mlp& net, int B, bool with_target, double* dis_host, double* l1_host, hipStream_t s) {
  stream_sync(s);
  const double* res = static_cast<const double*>(net.sout.h);
  std::memcpy(dis_host, res, B * sizeof(double));
  if (with_target && l1_host) std::memcpy(l1_host, res + B, B * sizeof(double));
}

void mlp_gradients(Mlp& net, const float* x_host, const float* y_host, int B, float* g_host, double* loss,
                   hipStream_t s) {
  alloc_train(net, B, s);
  stage_batch_input(net, x_host, B);
  DevBuf yb, lossp;
  h2d(yb, y_host, (size_t)B * net.dims[net.L], s);
  const int tiles = loss_tiles(net, B);
  lossp.reserve((size_t)net.E * tiles * 8);
  net.loss.reserve(net.E * 8);
  HIP_CHECK(hipMemsetAsync(net.g.p, 0, (size_t)net.E * net.P * 4, s));
  gather_batch(net, static_cast<const float*>(net.xin.d), nullptr, B, s);
  train_pass(net, B, yb.as<float>(), nullptr, lossp.as<double>(), nullptr, s);
  hipLaunchKernelGGL(loss_sum_kernel, dim3(net.E), dim3(64), 0, s, lossp.as<double>(), tiles,
                     (double)B * net.dims[net.L], net.loss.as<double>());
  HIP_CHECK(hipGetLastError());
  if (g_host) d2h(g_host, net.g.p, (size_t)net.E * net.P, s);
  if (loss) d2h(loss, net.loss.p, net.E, s);
  stream_sync(s);
}

void mlp_set_data(Mlp& net, const float* X, const float* Y, int64_t n, hipStream_t s) {
  h2d(net.dX, X, (size_t)n * net.dims[0], s);
  h2d(net.dY, Y, (size_t)n * net.dims[net.L], s);
  stream_sync(s);
  net.n_data = n;
}

void mlp_train(Mlp& net, const int32_t* batches, int steps, int B, float lr, float b1, float b2, float eps,
               double* losses, hipStream_t s) {
  alloc_train(net, B, s);
  DevBuf didx, lossp, lbuf;
  h2d(didx, batches, (size_t)steps * B, s);
  const int tiles = loss_tiles(net, B);
  // the tiles' sums of squares of up to 1 MiB of steps, summed into lbuf before
  // the next steps overwrite them
  const size_t step_bytes = (size_t)net.E * tiles * 8;
  const int group = (int)std::max<size_t>(1, std::min<size_t>(steps, (size_t(1) << 20) / step_bytes));
  lossp.reserve(group * step_bytes);
  lbuf.reserve((size_t)std::max(steps, 1) * net.E * 8);
  for (int it = 0; it < steps; ++it) {
    const int32_t* idx = didx.as<int32_t>() + (size_t)it * B;
    gather_batch(net, net.dX.as<float>(), idx, B, s);
    ++net.step;
    const AdamStep adam{lr, b1, b2, eps, 1.0f - powf(b1, (float)net.step), 1.0f - powf(b2, (float)net.step)};
    const int k = it % group;
    train_pass(net, B, net.dY.as<float>(), idx, lossp.as<double>() + (size_t)k * net.E * tiles, &adam, s);
    if (k + 1 == group || it + 1 == steps) {
      hipLaunchKernelGGL(loss_sum_kernel, dim3((k + 1) * net.E), dim3(64), 0, s, lossp.as<double>(), tiles,
                         (double)B * net.dims[net.L], lbuf.as<double>() + (size_t)(it - k) * net.E);
      HIP_CHECK(hipGetLastError());
    }
  }
  if (losses) d2h(losses, lbuf.p, (size_t)steps * net.E, s);
  stream_sync(s);
}

}  // namespace imped
