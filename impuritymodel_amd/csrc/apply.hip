// Operator application kernels: one lane per source product state.
//
// Replaces the inner loops of applyOp (impurityModel/ed/finite.py:1357-1388,
// 1415-1458) used by the Hamiltonian build (get_hamiltonian_matrix,
// finite.py:1585-1609), the BFS closure (expand_basis, finite.py:1737-1798)
// and transition operators (getSpectra, spectra.py:786).
//
// Each process (term) of an operator is compiled on the host to bit masks:
// it is non-zero on state s iff (s & care) == val, it maps s to s ^ flip, and
// its fermion sign is (-1)^(popcount(s & sgn) + parity) -- the product of the
// reference's sequential create/remove signs (create.py:142-148,
// remove.py:141-147).  Terms are grouped by flip mask: a group maps a source
// to exactly one target, so per-source duplicates merge inside the group in
// the operator dict's order, the order in which applyOp adds them.
//
// A wave handles 64 sources of one model, so the group/term loops are
// wave-uniform.  The term table streams through the wave's registers: lane i
// of a chunk holds term i's masks, value and sign data (one coalesced load
// per 64 terms, the next chunk's in flight while this one is used), and a
// term is broadcast to the wave by readlane.
#include "kernels.h"

namespace imped {

__device__ __forceinline__ bool key_eq(const uint64_t* a, const uint64_t* b, int W) {
  for (int w = 0; w < W; ++w)
    if (a[w] != b[w]) return false;
  return true;
}

__device__ __forceinline__ int32_t load_coherent(const int32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Look up (chain, key) in a table of pool ids; returns the id or HASH_EMPTY.
template <int W>
__device__ int32_t hash_find(const HashView& h, int32_t chain, const uint64_t* key) {
  uint32_t slot = hash_key((uint32_t)chain, key, W) & h.mask;
  for (;;) {
    const int32_t cur = h.table[slot];
    if (cur == HASH_EMPTY) return HASH_EMPTY;
    if (h.pool_chain[cur] == chain && key_eq(h.pool_keys + (size_t)cur * W, key, W)) return cur;
    slot = (slot + 1) & h.mask;
  }
}

constexpr int RESTR_LDS = 16;  // restrictions kept in LDS (more are read from memory)

// Index of the first of group_term_off[lo..hi] that is >= x (hi if none is
// smaller), searched 64 ways: every lane probes one position per round.
__device__ __forceinline__ int group_at_term(const int32_t* gto, int lo, int hi, int x, int lane) {
  while (lo < hi) {
    const int step = (hi - lo + 63) >> 6;
    const int idx = lo + lane * step;
    const int below = __popcll(__ballot(idx < hi && gto[idx] < x));  // a prefix of the lanes
    if (below == 0) break;
    const int up = lo + below * step;
    lo += (below - 1) * step + 1;
    hi = up < hi ? up : hi;
  }
  return __builtin_amdgcn_readfirstlane(lo);
}

__device__ __forceinline__ uint64_t lane_u64(uint64_t v, int i) {
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)v, i);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), i);
  return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ double lane_f64(double v, int i) {
  return __longlong_as_double((long long)lane_u64((uint64_t)__double_as_longlong(v), i));
}

// 64 terms, one per lane.  A state that matches has val on the care bits, so the
// part of its sign that those bits decide goes into the coefficient once, here
// (a negation is exact), and sgn keeps the other bits; terms without such bits, or
// without an imaginary part, skip that work by a wave-uniform bit test.
template <int W>
struct TermChunk {
  uint64_t care[W], val[W], sgn[W];
  double2 c;
  uint32_t meta;
  __device__ __forceinline__ void load(const OpsView& o, int t, int t_end) {
    if (t < t_end) {
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const uint64_t* m = o.term_masks + (size_t)t * 3 * W + w;
        care[w] = m[0];
        val[w] = m[W];
        sgn[w] = m[2 * W];
      }
      c = o.term_coef[t];
      meta = o.term_meta[t];
    }
  }
  // terms with sign bits left, terms with an imaginary part
  __device__ __forceinline__ void fold(uint64_t& has_sign, uint64_t& has_imag) {
    uint32_t par = meta & 1u;
    uint64_t left = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      par ^= (uint32_t)__popcll(val[w] & sgn[w]) & 1u;
      sgn[w] &= ~care[w];
      left |= sgn[w];
    }
    if (par) c = make_double2(-c.x, -c.y);
    has_sign = __ballot(left != 0);
    has_imag = __ballot(!(c.y == 0.0));
  }
};

// One wave per (64 sources, part of the model's groups): part p of a.split
// takes the groups whose terms start in the p-th equal share of the model's
// terms, and counts and offsets hold one value per (source, part), so the
// entries of a source stay in group order whatever the split is.
//
// What bounds it: instruction issue of the walk over the terms, 65 to 200 cycles a
// term.  Measured on 1000-term models, one launch: a few hundred sources 130 us with
// the terms in LDS and one wave per task, 45 us from registers with the groups
// divided, 24 us with the signs folded and the number operators' branches gone
// (they are one group of 340 matching terms, which stays with one wave); up to 3e6
// sources of two words 1.6, 1.1 and 0.95 ms.
template <int W, int MODE, bool FILL>
__global__ __launch_bounds__(256) void apply_kernel(ApplyArgs a) {
  __shared__ uint64_t l_rmask[4][RESTR_LDS * W];
  __shared__ int32_t l_rlohi[4][RESTR_LDS * 2];
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int64_t unit = (int64_t)blockIdx.x * (blockDim.x >> 6) + wv;
  const int64_t task_id = unit / a.split;
  const int part = __builtin_amdgcn_readfirstlane((int)(unit - task_id * a.split));
  if (task_id >= a.n_tasks) return;
  const WaveTask task = a.tasks[task_id];
  const int model = __builtin_amdgcn_readfirstlane(task.model);
  const int chain = __builtin_amdgcn_readfirstlane(task.chain);
  const int64_t src = task.begin + lane;
  const bool active = src < task.end;

  uint64_t s[W];
  for (int w = 0; w < W; ++w) s[w] = active ? a.src_keys[src * W + w] : 0ull;
  double2 amp = make_double2(1.0, 0.0);
  int32_t spos = 0;
  if (MODE == MODE_VECTOR && active) {
    amp = a.src_amps[src];
    spos = a.src_pos[src];
  }
  int64_t out = 0;
  int32_t cnt = 0;
  if (FILL && active) out = a.offsets[src * a.split + part];

  const OpsView& o = a.ops;
  int g0 = __builtin_amdgcn_readfirstlane(o.model_group_off[model]);
  int g1 = __builtin_amdgcn_readfirstlane(o.model_group_off[model + 1]);
  const int r0 = o.model_restr_off[model];
  const int r1 = o.model_restr_off[model + 1];
  if (a.split > 1) {
    const int tb = o.group_term_off[g0];
    const int64_t T = o.group_term_off[g1] - tb;
    const int lo = part > 0 ? group_at_term(o.group_term_off, g0, g1, tb + (int)(T * part / a.split), lane) : g0;
    const int hi =
        part + 1 < a.split ? group_at_term(o.group_term_off, g0, g1, tb + (int)(T * (part + 1) / a.split), lane) : g1;
    g0 = lo;
    g1 = hi;
  }
  int t = __builtin_amdgcn_readfirstlane(o.group_term_off[g0]);
  const int t_end = __builtin_amdgcn_readfirstlane(o.group_term_off[g1]);  // this wave's terms end here
  const int nr = r1 - r0;
  const int nrl = nr < RESTR_LDS ? nr : RESTR_LDS;
  uint64_t* lrm = l_rmask[wv];
  int32_t* lrl = l_rlohi[wv];
  if (MODE != MODE_FIXED) {
    for (int i = lane; i < nrl * W; i += 64) lrm[i] = o.restr_mask[(size_t)r0 * W + i];
    for (int i = lane; i < nrl * 2; i += 64) lrl[i] = o.restr_lohi[2 * r0 + i];
    // LDS writes by some lanes of the wave, read by every lane of it
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }

  TermChunk<W> cur{}, next{};
  int tc0 = t;  // first term of the chunk in registers
  uint64_t has_sign, has_imag;
  cur.load(o, tc0 + lane, t_end);
  next.load(o, tc0 + 64 + lane, t_end);
  cur.fold(has_sign, has_imag);
  int gc0 = g0;  // first group in registers
  int32_t gend = 0;
  uint64_t gflip[W] = {};
  auto load_groups = [&]() {
    if (gc0 + lane < g1) {
      gend = o.group_term_off[gc0 + lane + 1];
#pragma unroll
      for (int w = 0; w < W; ++w) gflip[w] = o.group_flip[(size_t)(gc0 + lane) * W + w];
    }
  };
  load_groups();

  for (int g = g0; g < g1; ++g) {
    if (g - gc0 == 64) {
      gc0 = g;
      load_groups();
    }
    const int te = __builtin_amdgcn_readlane(gend, g - gc0);
    double2 acc = make_double2(0.0, 0.0);
    bool any = false;
    int first = 0;
    // one matching term: add its signed value (in term order)
    auto take = [&](int i) {
      double cx = lane_f64(cur.c.x, i), cy = 0.0;
      if (has_imag >> i & 1) cy = lane_f64(cur.c.y, i);
      if (has_sign >> i & 1) {
        uint32_t par = 0;
#pragma unroll
        for (int w = 0; w < W; ++w) par ^= (uint32_t)__popcll(s[w] & lane_u64(cur.sgn[w], i)) & 1u;
        cx = par ? -cx : cx;
        cy = par ? -cy : cy;
      }
      acc.x += cx;
      if (has_imag >> i & 1) acc.y += cy;
      if (MODE == MODE_VECTOR && !any) first = (int)(__builtin_amdgcn_readlane(cur.meta, i) >> 1);
      any = true;
    };
    auto matches = [&](int i) {
      bool ok = true;
#pragma unroll
      for (int w = 0; w < W; ++w) ok = ok & ((s[w] & lane_u64(cur.care[w], i)) == lane_u64(cur.val[w], i));
      return ok;
    };
    while (t < te) {
      if (t - tc0 == 64) {
        tc0 = t;
        cur = next;
        next.load(o, tc0 + 64 + lane, t_end);
        cur.fold(has_sign, has_imag);
      }
      const int iend = te - tc0 < 64 ? te - tc0 : 64;
      int i = t - tc0;
      // Four mask tests at once, the matches taken in term order.  Where the four
      // are real and their signs are decided (number operators), adding 0 in the
      // lanes without a match takes the place of four branches; the sum is never
      // -0, so that adds nothing.
      for (; i + 4 <= iend; i += 4) {
        const bool k0 = matches(i), k1 = matches(i + 1), k2 = matches(i + 2), k3 = matches(i + 3);
        if (__ballot(k0 | k1 | k2 | k3) == 0) continue;
        if (MODE != MODE_VECTOR && ((has_sign | has_imag) >> i & 15) == 0) {
          const double c0 = lane_f64(cur.c.x, i), c1 = lane_f64(cur.c.x, i + 1);
          const double c2 = lane_f64(cur.c.x, i + 2), c3 = lane_f64(cur.c.x, i + 3);
          acc.x += k0 ? c0 : 0.0;
          acc.x += k1 ? c1 : 0.0;
          acc.x += k2 ? c2 : 0.0;
          acc.x += k3 ? c3 : 0.0;
          any = any | k0 | k1 | k2 | k3;
          continue;
        }
        if (k0) take(i);
        if (k1) take(i + 1);
        if (k2) take(i + 2);
        if (k3) take(i + 3);
      }
      for (; i < iend; ++i)
        if (matches(i)) take(i);
      t = tc0 + iend;
    }
    if (__ballot(any && active) == 0) continue;
    uint64_t tgt[W];
#pragma unroll
    for (int w = 0; w < W; ++w) tgt[w] = s[w] ^ lane_u64(gflip[w], g - gc0);
    if (!(any && active)) continue;
    bool keep = true;
    if (MODE != MODE_VECTOR) keep = abs2_ref(acc) >= a.weight_min;
    if (MODE != MODE_FIXED) {
      for (int r = 0; r < nrl && keep; ++r) {
        int n = 0;
#pragma unroll
        for (int w = 0; w < W; ++w) n += __popcll(tgt[w] & lrm[r * W + w]);
        keep = n >= lrl[2 * r] && n <= lrl[2 * r + 1];
      }
      for (int r = r0 + nrl; r < r1 && keep; ++r) {
        int n = 0;
#pragma unroll
        for (int w = 0; w < W; ++w) n += __popcll(tgt[w] & o.restr_mask[(size_t)r * W + w]);
        keep = n >= o.restr_lohi[2 * r] && n <= o.restr_lohi[2 * r + 1];
      }
    }
    int32_t local = 0;
    if (MODE == MODE_FIXED && keep) {
      int32_t id = hash_find<W>(a.hash, chain, tgt);
      keep = id >= 0;
      if (keep) local = a.pool_local[id];
    }
    if (!keep) continue;
    if (!FILL) {
      ++cnt;
      continue;
    }
    if (MODE == MODE_EXPAND) {
      // new targets are entered into the hash by discover_kernel afterwards
      for (int w = 0; w < W; ++w) a.out_keys[out * W + w] = tgt[w];
      a.out_val[out] = acc;
      a.out_chain[out] = chain;
    } else if (MODE == MODE_FIXED) {
      a.out_col[out] = local;
      a.out_val[out] = cconj(acc);
    } else {
      for (int w = 0; w < W; ++w) a.out_keys[out * W + w] = tgt[w];
      a.out_val[out] = cmul(amp, acc);
      a.out_vec[out] = chain;
      a.out_src[out] = spos;
      a.out_first[out] = first;
    }
    ++out;
  }
  if (!FILL && active) a.counts[src * a.split + part] = cnt;
}

template <int W>
static void launch_w(int mode, bool fill, const ApplyArgs& a, hipStream_t s) {
  const int threads = 256;
  const unsigned blocks = blocks_for(a.n_tasks * a.split, threads / 64);
  if (a.n_tasks == 0) return;
  TimedLaunch tl(fill ? "apply_fill" : "apply_count", s);
#define IMPED_LAUNCH(M, F) hipLaunchKernelGGL((apply_kernel<W, M, F>), dim3(blocks), dim3(threads), 0, s, a)
  if (mode == MODE_EXPAND) {
    if (fill) IMPED_LAUNCH(MODE_EXPAND, true); else IMPED_LAUNCH(MODE_EXPAND, false);
  } else if (mode == MODE_FIXED) {
    if (fill) IMPED_LAUNCH(MODE_FIXED, true); else IMPED_LAUNCH(MODE_FIXED, false);
  } else {
    if (fill) IMPED_LAUNCH(MODE_VECTOR, true); else IMPED_LAUNCH(MODE_VECTOR, false);
  }
#undef IMPED_LAUNCH
  HIP_CHECK(hipGetLastError());
}

// Every expand-fill entry e (chain[e], keys[e]) finds its state: a pool id, or
// the entry that entered the same (chain, key) into the table first in this
// launch (| CAND_FLAG), which is the layer's new state.  An entry's own number is
// its candidate id: the keys it is compared by were written by the launch before,
// so publishing a candidate is one compare-and-swap, with no key copy, fence or
// counter of its own, and the winners are compacted with one atomic per block.
// One thread per entry, so the dependent probes of many entries overlap.
//
// What bounds it: two to three random lines an entry (slot, key, chain) from
// memory once the table outgrows the caches.  The 12 layers that reach 2.9e6
// states of two words take 4.8 ms in all, 67 ms with a fenced key copy and two
// same-address counters per candidate.
template <int W>
__global__ __launch_bounds__(256) void discover_kernel(const uint64_t* keys, const int32_t* chain, int64_t E, HashView h,
                                                       int32_t* entry_id, int32_t* winner_slot, int32_t* winners,
                                                       int32_t* n_winners) {
  __shared__ int32_t wave_base[4];
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  bool won = false;
  if (e < E) {
    uint64_t k[W];
#pragma unroll
    for (int w = 0; w < W; ++w) k[w] = keys[e * W + w];
    const int32_t c = chain[e];
    uint32_t slot = hash_key((uint32_t)c, k, W) & h.mask;
    for (;;) {
      int32_t cur = load_coherent(&h.table[slot]);
      if (cur == HASH_EMPTY) {
        cur = atomicCAS(&h.table[slot], HASH_EMPTY, CAND_FLAG | (int32_t)e);
        if (cur == HASH_EMPTY) {
          won = true;
          winner_slot[e] = (int32_t)slot;
          entry_id[e] = CAND_FLAG | (int32_t)e;
          break;
        }
      }
      const bool cand = (cur & CAND_FLAG) != 0;
      const int32_t id = cur & ~CAND_FLAG;
      const uint64_t* q = (cand ? keys : h.pool_keys) + (size_t)id * W;
      const int32_t qc = (cand ? chain : h.pool_chain)[id];
      if (qc == c && key_eq(q, k, W)) {
        entry_id[e] = cur;
        break;
      }
      slot = (slot + 1) & h.mask;
    }
  }
  const uint64_t mask = __ballot(won);
  if (lane == 0) wave_base[wave] = __popcll(mask);
  __syncthreads();
  if (threadIdx.x == 0) {
    const int32_t n = wave_base[0] + wave_base[1] + wave_base[2] + wave_base[3];
    int32_t at = n > 0 ? atomicAdd(n_winners, n) : 0;
    for (int i = 0; i < 4; ++i) {
      const int32_t m = wave_base[i];
      wave_base[i] = at;
      at += m;
    }
  }
  __syncthreads();
  if (won) winners[wave_base[wave] + __popcll(mask & ((1ull << lane) - 1))] = (int32_t)e;
}

void launch_discover(int W, const uint64_t* keys, const int32_t* chain, int64_t E, HashView h, int32_t* entry_id,
                     int32_t* winner_slot, int32_t* winners, int32_t* n_winners, hipStream_t s) {
  if (E <= 0) return;
  TimedLaunch tl("discover", s);
  if (W == 1)
    hipLaunchKernelGGL(discover_kernel<1>, dim3(blocks_for(E, 256)), dim3(256), 0, s, keys, chain, E, h, entry_id,
                       winner_slot, winners, n_winners);
  else
    hipLaunchKernelGGL(discover_kernel<2>, dim3(blocks_for(E, 256)), dim3(256), 0, s, keys, chain, E, h, entry_id,
                       winner_slot, winners, n_winners);
  HIP_CHECK(hipGetLastError());
}

int apply_split(int64_t n_tasks) {
  int s = 1;
  while (s < kApplySplitMax && n_tasks * s < kApplySplitWaves) s *= 2;
  return s;
}

void launch_apply(int W, int mode, bool fill, const ApplyArgs& a, hipStream_t s) {
  if (W == 1)
    launch_w<1>(mode, fill, a, s);
  else
    launch_w<2>(mode, fill, a, s);
}

// ------------------------------------------------------------------ hash maintenance

__global__ void hash_clear_kernel(int32_t* t, uint32_t cap) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < cap) t[i] = HASH_EMPTY;
}

void launch_hash_clear(int32_t* table, uint32_t cap, hipStream_t s) {
  hipLaunchKernelGGL(hash_clear_kernel, dim3(blocks_for(cap, 256)), dim3(256), 0, s, table, cap);
  HIP_CHECK(hipGetLastError());
}

// Insert pool ids [first, first+count); ids are unique per (chain, key).
template <int W>
__global__ void hash_insert_pool_kernel(HashView h, int64_t first, int64_t count) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const int32_t id = (int32_t)(first + i);
  const uint64_t* key = h.pool_keys + (size_t)id * W;
  uint32_t slot = hash_key((uint32_t)h.pool_chain[id], key, W) & h.mask;
  for (;;) {
    int32_t prev = atomicCAS(&h.table[slot], HASH_EMPTY, id);
    if (prev == HASH_EMPTY) return;
    slot = (slot + 1) & h.mask;
  }
}

void launch_hash_insert_pool(int W, HashView h, int64_t first, int64_t count, hipStream_t s) {
  if (count == 0) return;
  if (W == 1)
    hipLaunchKernelGGL(hash_insert_pool_kernel<1>, dim3(blocks_for(count, 256)), dim3(256), 0, s, h, first, count);
  else
    hipLaunchKernelGGL(hash_insert_pool_kernel<2>, dim3(blocks_for(count, 256)), dim3(256), 0, s, h, first, count);
  HIP_CHECK(hipGetLastError());
}

}  // namespace imped
