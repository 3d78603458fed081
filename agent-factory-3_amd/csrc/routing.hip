// Token -> expert permutation (routing metadata) for the grouped expert GEMMs.
//
// Reference behaviour:
//   routing_replay   quantization.py:593-636: softmax over the K gathered
//                    logits of each token; stable sort of the flat [T*K]
//                    expert ids; gate_indx = inverse permutation; gate_scal =
//                    softmax weights in sorted order; hist = bincount.
//   top-k routing    quantization.py:551-590 (routing_torch_dist at world size
//                    1, the torch restatement of triton_kernels' routing):
//                    top-K logits per token by a stable descending sort (ties
//                    go to the lower expert id), softmax over those K, then
//                    the K (id, weight) pairs of a token sorted by expert id.
//   expt data        triton_kernels.routing.compute_expt_data_torch (called at
//                    quantization.py:588,627): token_offs_raw = exclusive scan
//                    of hist; per block size BM, token_offs_pad = exclusive
//                    scan of ceil(hist/BM) and block_pid_map[i] = (b<<16)|e for
//                    the b-th BM-row block of expert e, -1 for unused slots.
//
// The sort is a stable counting sort: histograms of chunks of the flat index,
// a scan over (expert, chunk), then a scatter where each entry's rank among
// equal ids earlier in its chunk keeps the order of the flat index.  Entries
// whose expert id is outside [0, E) are dropped (gate_indx = -1), the same
// shape the reference gives expert-parallel-masked entries.
//
// Up to 1024 experts the whole chain (ids and weights, sort, tile maps, work
// orders) is one launch of one block for small batches and three or four
// launches otherwise: every step is a few microseconds of latency, so what a call
// costs is the number of dependent steps, not bytes.  More experts take the older
// chain of one kernel per step.
#include <mutex>

#include "af3_common.h"

namespace {

constexpr int kChunk = 256;

__device__ __forceinline__ uint32_t bf16_bits_rne(float f) { return af3_f32_to_bf16(f); }

// one thread per token: ids/weights of its K slots (replay form)
__global__ void replay_token_kernel(const uint16_t* __restrict__ logits, int64_t ld, const int32_t* __restrict__ idx,
                                    int64_t T, int E, int K, int32_t* __restrict__ ids,
                                    uint16_t* __restrict__ scal) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= T) return;
  float v[16];
  int e[16];
  float mx = -INFINITY;
  for (int j = 0; j < K; ++j) {
    e[j] = idx[t * K + j];
    bool ok = e[j] >= 0 && e[j] < E;
    v[j] = ok ? af3_bf16_to_f32(logits[t * ld + e[j]]) : -INFINITY;
    mx = fmaxf(mx, v[j]);
  }
  float den = 0.f;
  for (int j = 0; j < K; ++j) {
    v[j] = (e[j] >= 0 && e[j] < E) ? expf(v[j] - mx) : 0.f;
    den += v[j];
  }
  for (int j = 0; j < K; ++j) {
    bool ok = e[j] >= 0 && e[j] < E;
    ids[t * K + j] = ok ? e[j] : -1;
    scal[t * K + j] = (uint16_t)bf16_bits_rne(v[j] / den);
  }
}

// one thread per token: top-K selection + softmax + sort of the K by expert id
__global__ void topk_token_kernel(const uint16_t* __restrict__ logits, int64_t ld, int64_t T, int E, int K,
                                  int32_t* __restrict__ ids, uint16_t* __restrict__ scal) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= T) return;
  float v[16];
  int e[16];
  for (int j = 0; j < K; ++j) {
    v[j] = -INFINITY;
    e[j] = E;  // sentinel larger than any id
  }
  const uint16_t* row = logits + t * ld;
  for (int x = 0; x < E; ++x) {
    float f = af3_bf16_to_f32(row[x]);
    // strict > keeps the earlier (lower) id on ties, matching a stable sort of -logits
    if (f > v[K - 1] || (e[K - 1] == E)) {
      int p = K - 1;
      while (p > 0 && (f > v[p - 1] || e[p - 1] == E)) {
        v[p] = v[p - 1];
        e[p] = e[p - 1];
        --p;
      }
      v[p] = f;
      e[p] = x;
    }
  }
  float mx = v[0];
  float w[16], den = 0.f;
  for (int j = 0; j < K; ++j) {
    w[j] = expf(v[j] - mx);
    den += w[j];
  }
  // softmax output is rounded to the logits dtype (bf16) before reordering
  uint16_t wb[16];
  for (int j = 0; j < K; ++j) wb[j] = (uint16_t)bf16_bits_rne(w[j] / den);
  // insertion sort of the K pairs by expert id (ids are distinct)
  for (int a = 1; a < K; ++a) {
    int ek = e[a];
    uint16_t wk = wb[a];
    int b = a - 1;
    while (b >= 0 && e[b] > ek) {
      e[b + 1] = e[b];
      wb[b + 1] = wb[b];
      --b;
    }
    e[b + 1] = ek;
    wb[b + 1] = wk;
  }
  for (int j = 0; j < K; ++j) {
    ids[t * K + j] = e[j];
    scal[t * K + j] = wb[j];
  }
}

// per-chunk histogram: counts[e * n_chunks + c]
__global__ void chunk_hist_kernel(const int32_t* __restrict__ ids, int64_t R, int E, int n_chunks,
                                  int32_t* __restrict__ counts) {
  extern __shared__ int32_t sh[];
  for (int e = threadIdx.x; e < E; e += blockDim.x) sh[e] = 0;
  __syncthreads();
  int64_t i = (int64_t)blockIdx.x * kChunk + threadIdx.x;
  if (i < R) {
    int e = ids[i];
    if (e >= 0) atomicAdd(&sh[e], 1);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += blockDim.x) counts[(int64_t)e * n_chunks + blockIdx.x] = sh[e];
}

// one block per expert: exclusive scan of its per-chunk counts (in place) and hist[e]
__global__ __launch_bounds__(256) void chunk_scan_kernel(int32_t* __restrict__ counts, int n_chunks,
                                                         int32_t* __restrict__ hist) {
  __shared__ int32_t sh[256];
  const int e = blockIdx.x, t = threadIdx.x;
  int32_t* row = counts + (int64_t)e * n_chunks;
  int32_t carry = 0;
  for (int base = 0; base < n_chunks; base += 256) {
    const int c = base + t;
    const int32_t v = c < n_chunks ? row[c] : 0;
    sh[t] = v;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
      int32_t add = t >= off ? sh[t - off] : 0;
      __syncthreads();
      sh[t] += add;
      __syncthreads();
    }
    if (c < n_chunks) row[c] = carry + sh[t] - v;
    carry += sh[255];
    __syncthreads();
  }
  if (t == 0) hist[e] = carry;
}

// single block: token_offs_raw = exclusive scan of hist over experts
__global__ __launch_bounds__(1024) void expert_scan_kernel(const int32_t* __restrict__ hist, int E,
                                                           int32_t* __restrict__ offs) {
  __shared__ int32_t sh[1024];
  const int t = threadIdx.x;
  int32_t carry = 0;
  for (int base = 0; base < E; base += 1024) {
    const int e = base + t;
    const int32_t v = e < E ? hist[e] : 0;
    sh[t] = v;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
      int32_t add = t >= off ? sh[t - off] : 0;
      __syncthreads();
      sh[t] += add;
      __syncthreads();
    }
    if (e < E) offs[e] = carry + sh[t] - v;
    carry += sh[1023];
    __syncthreads();
  }
  if (t == 0) offs[E] = carry;
}

// stable scatter of each chunk into expert-sorted order
__global__ void scatter_kernel(const int32_t* __restrict__ ids, const uint16_t* __restrict__ scal, int64_t R,
                               int n_chunks, const int32_t* __restrict__ offs, const int32_t* __restrict__ base,
                               int32_t* __restrict__ topk_indx,
                               int32_t* __restrict__ gate_indx, uint16_t* __restrict__ gate_scal) {
  __shared__ int32_t sid[kChunk];
  int64_t i = (int64_t)blockIdx.x * kChunk + threadIdx.x;
  int e = (i < R) ? ids[i] : -1;
  sid[threadIdx.x] = e;
  __syncthreads();
  if (i >= R) return;
  if (e < 0) {
    gate_indx[i] = -1;
    return;
  }
  int rank = 0;
  for (int j = 0; j < (int)threadIdx.x; ++j) rank += (sid[j] == e);
  int32_t pos = offs[e] + base[(int64_t)e * n_chunks + blockIdx.x] + rank;
  topk_indx[pos] = (int32_t)i;
  gate_indx[i] = pos;
  gate_scal[pos] = scal[i];
}

__global__ void zero_kernel(int32_t* __restrict__ p, int n) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0;
}

// sorted slots past the number of valid entries (only when some ids were dropped)
__global__ void fill_tail_kernel(const int32_t* __restrict__ offs, int E, int64_t R, int32_t* __restrict__ topk_indx,
                                 uint16_t* __restrict__ gate_scal) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= R) return;
  if (i >= offs[E]) {
    topk_indx[i] = -1;
    gate_scal[i] = 0;
  }
}

// ---------------------------------------------------------------------------
// Routing plan for E <= 1024 experts.
//
// What bounds it is a chain of short dependent steps, so the steps are merged:
//   * plan_small_kernel (T K <= 4096 entries): one block does everything;
//   * larger batches: token_hist_kernel (ids, weights, per-chunk histograms of
//     64 to 256 tokens), plan_scan_kernel (one block: prefix over chunks and
//     experts, tile maps, work orders), plan_scatter_kernel (stable scatter);
//   * past kPlanOneScan counts (what the scan's one block holds in registers at a
//     time) plan_prefix_kernel makes the prefix over the chunks first, 16
//     experts per block: one block walking the counts in groups of 8 took 70 us
//     of 92 at 131072 tokens over 128 experts.
// A token's 16 lanes hold its E logits (E <= 256) and pick the top K by K
// max-reductions of (order-preserving logit bits, inverted id) keys, so ties
// go to the lower id; one thread per token with a sorted insertion took
// 25-45 us (a serial pass over E with one wave per CU).  The rank of an entry
// among equal ids of its wave comes from ballots over the id's bits instead of
// a scan of the chunk.  Partial tiles are put in order by a counting sort of
// their sizes (comparing all pairs of experts took 540 us at 1024).  Measured (4
// of E, kernel time per call from ids and weights to the tile maps and work
// order, against one kernel per step): top-k of 23 tokens over 32 experts 51 ->
// 6.4 us, 4096 tokens 61 -> 16; replay of 1021 tokens over 128 experts 27 -> 15,
// 16384 tokens 30 -> 17, 131072 tokens 60 -> 47.
// ---------------------------------------------------------------------------
constexpr int kPlanMaxE = 1024;       // experts (one thread each in the scans)
constexpr int kPlanMaxTopkE = 256;    // experts of the 16-lane top-k (16 logits per lane)
constexpr int kPlanSmallR = 4096;     // entries of the one-block plan
constexpr int kPlanSmallTopkT = 256;  // tokens whose top-k the one-block plan takes along (64 per pass)
constexpr int kPlanSmallCnt = 16384;  // (64-entry group, expert) counters of the one-block plan (64 KB)
constexpr int kPlanTokens = 64;       // tokens of one pass of 16-lane groups (three-launch plan)
constexpr int kPlanMaxBm = 8;
constexpr int kPlanTails = 512;       // sizes of partial tiles sorted at a time
constexpr int kPlanSeg = 32;          // chunks per thread and round of the prefix over chunks (in registers)
constexpr int kPlanOneScan = 1024 * kPlanSeg;  // counts up to which plan_scan_kernel takes the prefix along
constexpr int kPlanPrefixE = 16;      // experts per block of the prefix kernel

// tile maps and work orders to make (n_bm = 0: none); orders for the first n_order sizes
struct PlanMaps {
  int n_bm, n_order, max_tiles;
  int bm[kPlanMaxBm];
  int32_t *offs_pad, *map, *order;  // [n_bm][E + 1], [n_bm][max_tiles], [n_order][max_tiles]
};

// bf16 bits -> 16-bit key in float order (-0 as +0; NaN lowest, as a stable descending sort puts it last)
__device__ __forceinline__ uint32_t plan_key16(uint32_t b) {
  if ((b & 0x7FFFu) > 0x7F80u) return 0u;
  if (b == 0x8000u) b = 0u;
  return (b & 0x8000u) ? (~b & 0xFFFFu) : (b | 0x8000u);
}
__device__ __forceinline__ float plan_key_value(uint32_t k16) {
  const uint32_t b = k16 == 0u ? 0x7FC0u : (k16 & 0x8000u) ? (k16 & 0x7FFFu) : (~k16 & 0xFFFFu);
  return af3_bf16_to_f32(b);
}

// The K (id, softmax weight) slots of token t by its 16 lanes (all 64 lanes of
// the wave must call it; t >= T is idle): lane j < K returns slot j's expert id
// (-1: dropped) and bf16 weight.  TOPK: slots by ascending id.
template <bool TOPK>
__device__ __forceinline__ void plan_token(const uint16_t* __restrict__ logits, int64_t ld,
                                           const int32_t* __restrict__ idx, int64_t t, int64_t T, int E, int K,
                                           int32_t& id, uint16_t& w) {
  const int l = threadIdx.x & 15;
  const bool on = t < T;
  float v = -INFINITY;
  int32_t e = -1;
  if constexpr (TOPK) {
    uint32_t key[kPlanMaxTopkE / 16];
    const uint16_t* row = logits + (on ? t : 0) * ld;
#pragma unroll
    for (int i = 0; i < kPlanMaxTopkE / 16; ++i) {
      const int x = l + 16 * i;
      key[i] = x < E ? (plan_key16(row[x]) << 16) | (0xFFFFu - (uint32_t)x) : 0u;
    }
    uint32_t mine = 0u;
    for (int j = 0; j < K; ++j) {
      uint32_t m = 0u;
#pragma unroll
      for (int i = 0; i < kPlanMaxTopkE / 16; ++i) m = max(m, key[i]);
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o, 16));
#pragma unroll
      for (int i = 0; i < kPlanMaxTopkE / 16; ++i) key[i] = key[i] == m ? 0u : key[i];
      if (l == j) mine = m;
    }
    v = plan_key_value(mine >> 16);
    e = (int32_t)(0xFFFFu - (mine & 0xFFFFu));
  } else if (on && l < K) {
    e = idx[t * K + l];
    if (e < 0 || e >= E)
      e = -1;
    else
      v = af3_bf16_to_f32(logits[t * ld + e]);
  }
  float mx = TOPK ? __shfl(v, 0, 16) : -INFINITY;
  if constexpr (!TOPK)
    for (int j = 0; j < K; ++j) mx = fmaxf(mx, __shfl(v, j, 16));
  const float x = e >= 0 ? expf(v - mx) : 0.f;
  float den = 0.f;
  for (int j = 0; j < K; ++j) den += __shfl(x, j, 16);  // in slot order
  uint32_t wb = bf16_bits_rne(x / den);
  if constexpr (TOPK) {  // by ascending id: slot of winner j = winners with a lower id
    int rank = 0;
    for (int j = 0; j < K; ++j) rank += __shfl(e, j, 16) < e;
    int32_t se = -1;
    uint32_t sw = 0u;
    for (int j = 0; j < K; ++j) {
      const int r = __shfl(rank, j, 16);
      const int32_t ej = __shfl(e, j, 16);
      const uint32_t wj = (uint32_t)__shfl((int)wb, j, 16);
      if (r == l) {
        se = ej;
        sw = wj;
      }
    }
    e = se;
    wb = sw;
  }
  id = e;
  w = (uint16_t)wb;
}

// rank of this lane's id among the equal ids of lower lanes, and how many lanes hold it (e < 0: none)
__device__ __forceinline__ int plan_wave_rank(int e, int ebits, int& count) {
  uint64_t m = __ballot(e >= 0);
  for (int b = 0; b < ebits; ++b) {
    const uint64_t s = __ballot((e >> b) & 1);
    m &= ((e >> b) & 1) ? s : ~s;
  }
  const int lane = threadIdx.x & 63;
  count = __popcll(m);
  return __popcll(m & ((1ull << lane) - 1ull));
}

// inclusive prefix over a wave, all lanes active: within rows of 16 lanes, then the
// last lane of rows 0 and 2 into the next row, then lane 31 into the upper half
// (a step is one instruction; six shuffles through the LDS unit took ten times it)
__device__ __forceinline__ int plan_wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return v;
}
// the last lane's value
__device__ __forceinline__ int plan_wave_last(int v) { return __builtin_amdgcn_readlane(v, 63); }

__device__ __forceinline__ int plan_wave_sum(int v) { return plan_wave_last(plan_wave_scan(v)); }

// order j's partial tiles, after the full ones, by decreasing rows (ties to the
// lower expert): a counting sort of the tails by one wave, kPlanTails sizes at a
// time from the largest (cnt: LDS), then the -1 padding
__device__ void plan_tail_order(const PlanMaps& m, int j, int E, const int32_t* counts, int32_t* cnt) {
  const int lane = threadIdx.x & 63, bm = m.bm[j];
  int32_t* const out = m.order + (int64_t)j * m.max_tiles;
  int at = 0;
  for (int e = lane; e < E; e += 64) at += counts[e] / bm;
  at = plan_wave_sum(at);  // full tiles
  const auto sync = [] {  // orders the wave's LDS accesses
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  for (int hi = bm; hi > 1; hi -= kPlanTails) {  // tails in [lo, hi), keys hi - 1 - tail
    const int lo = max(hi - kPlanTails, 1), n_keys = hi - lo;
    const int bits = n_keys > 1 ? 32 - __clz(n_keys - 1) : 1;
    for (int i = lane; i < n_keys; i += 64) cnt[i] = 0;
    sync();
    for (int e = lane; e < E; e += 64) {
      const int tail = counts[e] % bm;
      if (tail >= lo && tail < hi) atomicAdd(&cnt[hi - 1 - tail], 1);
    }
    sync();
    for (int i0 = 0; i0 < n_keys; i0 += 64) {
      const int v = i0 + lane < n_keys ? cnt[i0 + lane] : 0;
      const int incl = plan_wave_scan(v);
      if (i0 + lane < n_keys) cnt[i0 + lane] = at + incl - v;
      at += plan_wave_last(incl);
    }
    sync();
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + lane, h = e < E ? counts[e] : 0;
      const int full = h / bm, tail = h - full * bm;
      const int key = tail >= lo && tail < hi ? hi - 1 - tail : -1;
      int c;
      const int rank = plan_wave_rank(key, bits, c);
      const int pos = key >= 0 ? cnt[key] + rank : m.max_tiles;
      if (pos < m.max_tiles) out[pos] = (full << 16) | e;
      sync();
      if (key >= 0 && rank == 0) cnt[key] += c;
      sync();
    }
  }
  for (int i = at + lane; i < m.max_tiles; i += 64) out[i] = -1;
}

// padded offsets, tile maps and work orders from the experts' counts (LDS, E
// ints, published by a barrier).  A block of one CU issues one wave instruction
// per SIMD and cycle, so nothing is run by 16 waves that one needs once: a wave
// makes one order's partial tiles, or the (full) tiles of one map or order for as
// large a part of the experts as leaves every wave a job.
__device__ void plan_maps(const PlanMaps& m, int E, const int32_t* counts, int32_t* tails) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_grp = (E + 63) >> 6, n_out = m.n_bm + m.n_order;
  if (n_out == 0) return;
  if (wave < m.n_order) plan_tail_order(m, wave, E, counts, tails + wave * kPlanTails);
  const int parts = min(max((16 - m.n_order) / n_out, 1), n_grp), per = (n_grp + parts - 1) / parts;
  const int first = wave < m.n_order ? wave + 16 : wave;  // (more jobs than waves: n_out > 8)
  for (int job = first - m.n_order; job < n_out * parts; job += 16) {
    const int which = job / parts, part = job % parts;
    const bool ord = which >= m.n_bm;
    const int b = ord ? which - m.n_bm : which;
    const int bm = m.bm[b], up = ord ? 0 : bm - 1;
    int32_t* const out = (ord ? m.order : m.map) + (int64_t)b * m.max_tiles;
    const int g_end = min(n_grp, (part + 1) * per);
    int base = 0;  // tiles of the experts before the group
    if (part > 0) {
      for (int f = lane; f < min(64 * part * per, E); f += 64) base += (counts[f] + up) / bm;
      base = plan_wave_sum(base);
    }
    for (int grp = part * per; grp < g_end; ++grp) {
      const int e = 64 * grp + lane, h = e < E ? counts[e] : 0;
      const int n = (h + up) / bm;
      const int incl = plan_wave_scan(n), at = base + incl - n;
      if (!ord && e < E) m.offs_pad[b * (E + 1) + e] = at;
      // an expert's first tiles by its lane, the rest by the wave
      constexpr int kOwn = 8;
      for (int i = 0; i < kOwn && __ballot(i < n); ++i)
        if (i < n && at + i < m.max_tiles) out[at + i] = (i << 16) | e;
      for (uint64_t big = __ballot(n > kOwn); big; big &= big - 1) {
        const int l = __ffsll((unsigned long long)big) - 1;
        const int n_l = __shfl(n, l, 64), at_l = __shfl(at, l, 64);
        for (int i = kOwn + lane; i < n_l; i += 64)
          if (at_l + i < m.max_tiles) out[at_l + i] = (i << 16) | (64 * grp + l);
      }
      base += plan_wave_last(incl);
    }
    if (!ord && g_end == n_grp && part * per < n_grp) {  // the part with the last group
      if (lane == 0) m.offs_pad[b * (E + 1) + E] = base;
      for (int i = base + lane; i < m.max_tiles; i += 64) out[i] = -1;
    }
  }
}

// hist, offs [E + 1] and start (LDS) = the exclusive prefix of the experts' counts (LDS), by one wave; returns the sum
__device__ __forceinline__ int plan_offsets(int E, int32_t* counts, int32_t* __restrict__ hist,
                                            int32_t* __restrict__ offs, int32_t* start) {
  const int lane = threadIdx.x & 63;
  int carry = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int e = e0 + lane, h = e < E ? counts[e] : 0;
    const int incl = plan_wave_scan(h);
    if (e < E) {
      hist[e] = h;
      offs[e] = carry + incl - h;
      start[e] = carry + incl - h;
    }
    carry += plan_wave_last(incl);
  }
  if (lane == 0) offs[E] = carry;
  return carry;
}

// the whole plan in one block. MODE 0: top-k of the logits, 1: given ids, 2: ids / weights already made
template <int MODE>
__global__ __launch_bounds__(1024) void plan_small_kernel(const uint16_t* __restrict__ logits, int64_t ld,
                                                          const int32_t* __restrict__ idx, int T, int E, int K,
                                                          const int32_t* __restrict__ ids_in,
                                                          const uint16_t* __restrict__ scal_in, int ebits,
                                                          uint16_t* __restrict__ gate_scal, int32_t* __restrict__ hist,
                                                          int32_t* __restrict__ topk_indx,
                                                          int32_t* __restrict__ gate_indx, int32_t* __restrict__ offs,
                                                          PlanMaps m) {
  __shared__ int32_t ids[kPlanSmallR];
  __shared__ uint16_t sc[kPlanSmallR];
  __shared__ int32_t cnt[kPlanSmallCnt];  // [64-entry group][E]
  __shared__ int32_t start[kPlanMaxE];
  __shared__ int32_t counts[kPlanMaxE];
  __shared__ int32_t total;
  __shared__ int32_t tails[kPlanMaxBm * kPlanTails];
  const int t = threadIdx.x, R = T * K, ngroup = (R + 63) / 64;
  if constexpr (MODE == 2) {
    for (int i = t; i < R; i += 1024) {
      ids[i] = ids_in[i];
      sc[i] = scal_in[i];
    }
  } else if constexpr (MODE == 0) {
    for (int t0 = 4 * (t >> 6); t0 < T; t0 += 64) {  // four tokens per wave, idle waves skip
      const int tok = t0 + ((t & 63) >> 4);
      int32_t e;
      uint16_t w;
      plan_token<true>(logits, ld, idx, tok, T, E, K, e, w);
      if (tok < T && (t & 15) < K) {
        ids[tok * K + (t & 15)] = e;
        sc[tok * K + (t & 15)] = w;
      }
    }
  } else {
    // replay: every slot's id, then every slot's logit (two loads deep however
    // many tokens), then one thread per token
    float* const val = (float*)cnt;
    int32_t id[kPlanSmallR / 1024];
#pragma unroll
    for (int q = 0; q < kPlanSmallR / 1024; ++q) {
      const int i = q * 1024 + t;
      id[q] = i < R ? idx[i] : -1;
    }
#pragma unroll
    for (int q = 0; q < kPlanSmallR / 1024; ++q) {
      const int i = q * 1024 + t;
      const bool ok = id[q] >= 0 && id[q] < E;
      const float v = ok ? af3_bf16_to_f32(logits[(int64_t)(i / K) * ld + id[q]]) : -INFINITY;
      if (i < R) {
        ids[i] = ok ? id[q] : -1;
        val[i] = v;
      }
    }
    __syncthreads();
    for (int tok = t; tok < T; tok += 1024) {
      float mx = -INFINITY, den = 0.f;
      for (int j = 0; j < K; ++j) mx = fmaxf(mx, val[tok * K + j]);
      for (int j = 0; j < K; ++j) {
        const float x = ids[tok * K + j] >= 0 ? expf(val[tok * K + j] - mx) : 0.f;
        val[tok * K + j] = x;
        den += x;
      }
      for (int j = 0; j < K; ++j) sc[tok * K + j] = (uint16_t)bf16_bits_rne(val[tok * K + j] / den);
    }
    __syncthreads();
  }
  for (int i = t; i < ngroup * E; i += 1024) cnt[i] = 0;
  __syncthreads();
  int rank[kPlanSmallR / 1024];
#pragma unroll
  for (int q = 0; q < kPlanSmallR / 1024; ++q) {
    const int i = q * 1024 + t;
    rank[q] = 0;
    if (q * 1024 + (t & ~63) >= R) continue;  // wave-uniform
    const int e = i < R ? ids[i] : -1;
    int c;
    rank[q] = plan_wave_rank(e, ebits, c);
    if (e >= 0 && rank[q] == 0) cnt[(i >> 6) * E + e] = c;
  }
  __syncthreads();
  for (int e = t; e < E; e += 1024) {
    int h = 0;
    for (int g = 0; g < ngroup; g += 8) {
      int c[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) c[j] = g + j < ngroup ? cnt[(g + j) * E + e] : 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (g + j < ngroup) cnt[(g + j) * E + e] = h;
        h += c[j];
      }
    }
    counts[e] = h;
  }
  __syncthreads();
  if (t < 64) {
    const int n = plan_offsets(E, counts, hist, offs, start);
    if (t == 0) total = n;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kPlanSmallR / 1024; ++q) {
    const int i = q * 1024 + t;
    if (i >= R) continue;
    const int e = ids[i];
    if (e >= 0) {
      const int pos = start[e] + cnt[(i >> 6) * E + e] + rank[q];
      topk_indx[pos] = i;
      gate_indx[i] = pos;
      gate_scal[pos] = sc[i];
    } else {
      gate_indx[i] = -1;
    }
    if (i >= total) {  // slots past the valid entries
      topk_indx[i] = -1;
      gate_scal[i] = 0;
    }
  }
  plan_maps(m, E, counts, tails);
}

// ids and weights (MODE as above) and the expert counts of each chunk of `chunk` tokens: counts[chunk][E]
template <int MODE>
__global__ __launch_bounds__(1024) void token_hist_kernel(const uint16_t* __restrict__ logits, int64_t ld,
                                                          const int32_t* __restrict__ idx, int64_t T, int E, int K,
                                                          int chunk, int32_t* __restrict__ ids,
                                                          uint16_t* __restrict__ scal, int32_t* __restrict__ counts) {
  __shared__ int32_t sh[kPlanMaxE];
  const int t = threadIdx.x;
  for (int e = t; e < E; e += 1024) sh[e] = 0;
  __syncthreads();
  const int64_t t0 = (int64_t)blockIdx.x * chunk;
  if constexpr (MODE == 2) {
    const int64_t hi = min((t0 + chunk) * K, T * K);
    for (int64_t i = t0 * K + t; i < hi; i += 1024)
      if (ids[i] >= 0) atomicAdd(&sh[ids[i]], 1);
  } else {
    for (int q = 0; q < chunk; q += kPlanTokens) {
      const int64_t tok = t0 + q + (t >> 4);
      int32_t e;
      uint16_t w;
      plan_token<MODE == 0>(logits, ld, idx, tok, T, E, K, e, w);
      if (tok < T && (t & 15) < K) {
        ids[tok * K + (t & 15)] = e;
        scal[tok * K + (t & 15)] = w;
        if (e >= 0) atomicAdd(&sh[e], 1);
      }
    }
  }
  __syncthreads();
  for (int e = t; e < E; e += 1024) counts[(int64_t)blockIdx.x * E + e] = sh[e];
}

// counts[chunk][e] -> their exclusive prefix over the chunks, in place; returns
// the sum.  `width` (a power of two) threads side by side take as many experts,
// the block's 1024 / width segments of them kPlanSeg chunks each: a round's counts
// are read once, all in flight together, and held for the write.
__device__ int plan_prefix(int32_t* __restrict__ counts, int n_chunks, int E, int e, int width, int32_t* seg_sum) {
  const int t = threadIdx.x, x = t & (width - 1), seg = t / width, nseg = 1024 / width;
  int32_t* const col = counts + min(e, E - 1);
  int carry = 0;
  for (int b0 = 0; b0 < n_chunks; b0 += nseg * kPlanSeg) {
    const int per = min(kPlanSeg, (n_chunks - b0 + nseg - 1) / nseg);
    const int c0 = b0 + seg * per, n = e < E ? min(per, n_chunks - c0) : 0;  // n < 0: none
    int u[kPlanSeg];
#pragma unroll
    for (int j0 = 0; j0 < kPlanSeg; j0 += 8)
      if (j0 < per) {
#pragma unroll
        for (int j = j0; j < j0 + 8; ++j) u[j] = col[(int64_t)min(c0 + j, n_chunks - 1) * E];
      }
    int sum = 0;
#pragma unroll
    for (int j0 = 0; j0 < kPlanSeg; j0 += 8)
      if (j0 < per) {
#pragma unroll
        for (int j = j0; j < j0 + 8; ++j) {
          u[j] = j < n ? u[j] : 0;
          sum += u[j];
        }
      }
    seg_sum[t] = sum;
    __syncthreads();
    int run = carry, all = 0;
#pragma unroll 4
    for (int s = 0; s < nseg; ++s) {
      const int v = seg_sum[s * width + x];
      run += s < seg ? v : 0;
      all += v;
    }
#pragma unroll
    for (int j0 = 0; j0 < kPlanSeg; j0 += 8)
      if (j0 < per) {
#pragma unroll
        for (int j = j0; j < j0 + 8; ++j) {
          if (j < n) col[(int64_t)(c0 + j) * E] = run;
          run += u[j];
        }
      }
    carry += all;
    __syncthreads();
  }
  return carry;
}

// the prefix over the chunks of kPlanPrefixE experts per block, and hist
__global__ __launch_bounds__(1024) void plan_prefix_kernel(int32_t* __restrict__ counts, int n_chunks, int E,
                                                           int32_t* __restrict__ hist) {
  __shared__ int32_t seg_sum[1024];
  const int t = threadIdx.x, e = blockIdx.x * kPlanPrefixE + (t & (kPlanPrefixE - 1));
  const int all = plan_prefix(counts, n_chunks, E, e, kPlanPrefixE, seg_sum);
  if (t < kPlanPrefixE && e < E) hist[e] = all;
}

// one block: counts[chunk][E] -> exclusive prefix over the chunks (n_chunks 0:
// done, hist holds the sums), then hist, offs, tile maps and orders
__global__ __launch_bounds__(1024) void plan_scan_kernel(int32_t* __restrict__ counts, int n_chunks, int E, int epad,
                                                         int32_t* __restrict__ hist, int32_t* __restrict__ offs,
                                                         PlanMaps m) {
  __shared__ int32_t cnt[kPlanMaxE];
  __shared__ int32_t start[kPlanMaxE];
  __shared__ int32_t scratch[kPlanMaxBm * kPlanTails];
  static_assert(kPlanMaxBm * kPlanTails >= 1024, "the segments' sums, then the tails");
  const int t = threadIdx.x;
  if (n_chunks > 0) {
    const int all = plan_prefix(counts, n_chunks, E, t & (epad - 1), epad, scratch);
    if (t < E) cnt[t] = all;  // threads 0 .. E - 1 are segment 0
  } else if (t < E) {
    cnt[t] = hist[t];
  }
  __syncthreads();
  if (t >= 960) plan_offsets(E, cnt, hist, offs, start);  // the last wave, the maps by the others
  plan_maps(m, E, cnt, scratch);
}

// stable scatter of chunk blockIdx.x into expert-sorted order, and the slots past the valid entries
__global__ __launch_bounds__(256) void plan_scatter_kernel(const int32_t* __restrict__ ids,
                                                            const uint16_t* __restrict__ scal, int64_t R, int E,
                                                            int chunk_entries, int ebits,
                                                            const int32_t* __restrict__ offs,
                                                            const int32_t* __restrict__ counts,
                                                            int32_t* __restrict__ topk_indx,
                                                            int32_t* __restrict__ gate_indx,
                                                            uint16_t* __restrict__ gate_scal) {
  __shared__ int32_t base[kPlanMaxE];
  __shared__ int32_t cnt[4 * kPlanMaxE];  // [wave][E] of one pass of 256 entries
  const int t = threadIdx.x, wave = t >> 6;
  for (int e = t; e < E; e += 256) base[e] = offs[e] + counts[(int64_t)blockIdx.x * E + e];
  const int64_t valid = offs[E];
  const int64_t lo = (int64_t)blockIdx.x * chunk_entries;
  const int64_t hi = min(lo + chunk_entries, R);
  for (int64_t i0 = lo; i0 < hi; i0 += 256) {
    const int64_t i = i0 + t;
    const int e = i < hi ? ids[i] : -1;
    for (int q = t; q < 4 * E; q += 256) cnt[q] = 0;
    __syncthreads();
    int c;
    const int rank = plan_wave_rank(e, ebits, c);
    if (e >= 0 && rank == 0) cnt[wave * E + e] = c;
    __syncthreads();
    for (int x = t; x < E; x += 256) {
      const int c0 = cnt[x], c1 = cnt[E + x], c2 = cnt[2 * E + x], c3 = cnt[3 * E + x], b0 = base[x];
      cnt[x] = b0;
      cnt[E + x] = b0 + c0;
      cnt[2 * E + x] = b0 + c0 + c1;
      cnt[3 * E + x] = b0 + c0 + c1 + c2;
      base[x] = b0 + c0 + c1 + c2 + c3;
    }
    __syncthreads();
    if (i < hi) {
      if (e >= 0) {
        const int pos = cnt[wave * E + e] + rank;
        topk_indx[pos] = (int32_t)i;
        gate_indx[i] = pos;
        gate_scal[pos] = scal[i];
      } else {
        gate_indx[i] = -1;
      }
      if (i >= valid) {
        topk_indx[i] = -1;
        gate_scal[i] = 0;
      }
    }
    __syncthreads();
  }
}

// ---- expert data: padded tile offsets and block -> (block, expert) map -----
// per tile size (one 1024-thread block each): the exclusive prefix of the
// experts' tile counts -> offs_pad, then the tile -> (expert, tile) map
constexpr int kScanMaxE = 4096;

__global__ __launch_bounds__(1024) void tile_scan_map_kernel(const int32_t* __restrict__ hist, int E,
                                                             const int32_t* __restrict__ block_ms, int max_tiles,
                                                             int32_t* __restrict__ offs_pad /* n_bm x (E+1) */,
                                                             int32_t* __restrict__ map /* n_bm x max_tiles */) {
  __shared__ int32_t op[kScanMaxE + 1];
  __shared__ int32_t part[1024];
  const int b = blockIdx.x, t = threadIdx.x;
  const int bm = block_ms[b];
  // thread t owns experts [t * per, (t + 1) * per)
  const int per = (E + 1023) / 1024;
  int32_t run = 0;
  for (int i = 0; i < per; ++i) {
    const int e = t * per + i;
    if (e < E) {
      const int32_t n = (hist[e] + bm - 1) / bm;
      op[e] = n;
      run += n;
    }
  }
  part[t] = run;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const int32_t v = t >= off ? part[t - off] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  int32_t pos = part[t] - run;
  for (int i = 0; i < per; ++i) {
    const int e = t * per + i;
    if (e < E) {
      const int32_t n = op[e];
      op[e] = pos;
      pos += n;
    }
  }
  if (t == 1023) op[E] = part[1023];
  __syncthreads();
  for (int e = t; e <= E; e += 1024) offs_pad[b * (E + 1) + e] = op[e];
  for (int i = t; i < max_tiles; i += 1024) {
    int32_t val = -1;
    if (i < op[E]) {
      // largest e with op[e] <= i (experts with zero tiles have op[e] == op[e+1])
      int lo = 0, hi = E - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (op[mid] <= i)
          lo = mid;
        else
          hi = mid - 1;
      }
      val = ((i - op[lo]) << 16) | lo;
    }
    map[(int64_t)b * max_tiles + i] = val;
  }
}

// ---- grouped-GEMM tile order: full tiles first (expert order), then the
// experts' partial last tiles by decreasing row count (ties: lower expert first)
constexpr int kSchedMaxE = 4096;
constexpr int kSchedMaxBM = 512;

__global__ __launch_bounds__(1024) void tile_order_kernel(const int32_t* __restrict__ hist, int E, int bm,
                                                          int max_tiles, int32_t* __restrict__ order) {
  __shared__ int32_t nfull[kSchedMaxE];
  __shared__ int32_t tail[kSchedMaxE];
  __shared__ int32_t start[kSchedMaxBM + 1];  // tails of size s start at start[s]
  __shared__ int32_t part[1024];               // prefix of full-tile counts
  __shared__ int32_t suf[1024];                // suffix of the tail-size histogram
  const int t = threadIdx.x;
  for (int e = t; e < E; e += 1024) {
    const int h = hist[e];
    nfull[e] = h / bm;
    tail[e] = h % bm;
  }
  for (int s = t; s <= kSchedMaxBM; s += 1024) start[s] = 0;
  __syncthreads();
  for (int e = t; e < E; e += 1024)
    if (tail[e]) atomicAdd(&start[tail[e]], 1);
  // exclusive prefix of full-tile counts over experts: thread t owns experts
  // [t * per, (t + 1) * per)
  const int per = (E + 1023) / 1024;
  int32_t run = 0;
  for (int i = 0; i < per; ++i) {
    const int e = t * per + i;
    if (e < E) run += nfull[e];
  }
  part[t] = run;
  __syncthreads();
  // thread t holds the count of tail size t (sizes 1 .. bm - 1; bm <= 1024)
  const int32_t cnt = (t >= 1 && t < bm) ? start[t] : 0;
  suf[t] = cnt;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const int32_t v = t >= off ? part[t - off] : 0;
    const int32_t w = t + off < 1024 ? suf[t + off] : 0;
    __syncthreads();
    part[t] += v;
    suf[t] += w;
    __syncthreads();
  }
  const int32_t total_full = part[1023];
  const int32_t n_tiles = total_full + suf[0];  // full tiles + one partial tile per expert with a tail
  // partial tiles by decreasing size: size s starts after every larger one
  if (t >= 1 && t < bm) start[t] = suf[t] - cnt;
  __syncthreads();
  int32_t pos = part[t] - run;
  for (int i = 0; i < per; ++i) {
    const int e = t * per + i;
    if (e >= E) break;
    // (a max_tiles below the real tile count truncates the order instead of
    // writing past it)
    for (int b = 0; b < nfull[e]; ++b)
      if (pos + b < max_tiles) order[pos + b] = (b << 16) | e;
    pos += nfull[e];
    const int s = tail[e];
    if (s) {
      int rank = start[s];
      for (int f = 0; f < e; ++f) rank += tail[f] == s;
      if (total_full + rank < max_tiles) order[total_full + rank] = (nfull[e] << 16) | e;
    }
  }
  for (int i = n_tiles + t; i < max_tiles; i += 1024) order[i] = -1;
}

}  // namespace

// What a batch keeps in the workspace: ids [R] at 0, weights [R], then one row
// of E counts per chunk.  The size queries and the launches both take it from
// here.  A chunk of the plan holds at least as many entries as the older
// chain's kChunk (64 tokens of 4 entries or more, 128 of 2 or 3, 256 of one), so
// the plan never needs more than the older chain did.
struct RoutingLayout {
  int chunk_tokens;  // tokens per chunk (plan)
  int64_t rows;      // chunks
  size_t scal, counts, bytes;
};
static RoutingLayout routing_layout(int64_t T, int E, int K) {
  const int64_t R = T * K;
  const auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
  RoutingLayout l;
  l.chunk_tokens = kPlanTokens * (K >= 4 ? 1 : K >= 2 ? 2 : 4);
  l.rows = E <= kPlanMaxE ? af3_cdiv(T, l.chunk_tokens) : af3_cdiv(R, kChunk);
  l.scal = up((size_t)R * 4);
  l.counts = up(l.scal + (size_t)R * 2);
  l.bytes = l.counts + (size_t)l.rows * E * 4 + 256;
  return l;
}

extern "C" size_t af3_routing_workspace_bytes(int64_t n_tokens, int n_expts_tot, int n_expts_act) {
  return routing_layout(n_tokens, n_expts_tot, n_expts_act).bytes;
}

extern "C" size_t af3_routing_count_rows(int64_t n_tokens, int n_expts_tot, int n_expts_act) {
  return (size_t)routing_layout(n_tokens, n_expts_tot, n_expts_act).rows;
}

extern "C" size_t af3_routing_plan_workspace_bytes(int64_t n_tokens, int n_expts_tot, int n_expts_act, int topk);

// whether the one-block plan takes the batch: replayed ids are one load per
// slot, the top-k of more than a few passes of tokens goes over more blocks
static bool plan_one_block(bool topk, int64_t T, int E, int K) {
  const int64_t R = T * K;
  return E <= kPlanMaxE && R <= kPlanSmallR && af3_cdiv(R, 64) * E <= kPlanSmallCnt &&
         (!topk || E > kPlanMaxTopkE || T <= kPlanSmallTopkT);
}

// E <= 1024: the merged chain, with the tile maps of `m` where it asks for any
static int routing_plan(bool topk, const uint16_t* logits, int64_t ld, const int32_t* expt_indx, int64_t T, int E, int K,
                        uint16_t* gate_scal, int32_t* hist, int32_t* topk_indx, int32_t* gate_indx,
                        int32_t* token_offs_raw, int32_t* ids, uint16_t* scal, int32_t* counts,
                        const RoutingLayout& lay, const PlanMaps& m, hipStream_t stream) {
  const int64_t R = T * K;
  const int ebits = E > 1 ? 32 - __builtin_clz((unsigned)(E - 1)) : 1;
  const bool lane_topk = topk && E <= kPlanMaxTopkE;
  if (topk && !lane_topk && T > 0) {
    hipLaunchKernelGGL(topk_token_kernel, dim3((unsigned)af3_cdiv(T, 128)), dim3(128), 0, stream, logits, ld, T, E, K,
                       ids, scal);
    int rc = af3::check_launch("routing/token");
    if (rc) return rc;
  }
  const int mode = !topk ? 1 : lane_topk ? 0 : 2;
  static_assert(kPlanSmallR <= kPlanSmallCnt, "the counters' other use");
  if (plan_one_block(topk, T, E, K)) {
#define AF3_PLAN(md)                                                                                                 \
  hipLaunchKernelGGL(plan_small_kernel<md>, dim3(1), dim3(1024), 0, stream, logits, ld, expt_indx, (int)T, E, K, ids, \
                     scal, ebits, gate_scal, hist, topk_indx, gate_indx, token_offs_raw, m)
    if (mode == 0) AF3_PLAN(0);
    else if (mode == 1) AF3_PLAN(1);
    else AF3_PLAN(2);
#undef AF3_PLAN
    return af3::check_launch("routing/plan");
  }
  const int n_chunks = (int)lay.rows;
#define AF3_TOK(md)                                                                                          \
  hipLaunchKernelGGL(token_hist_kernel<md>, dim3(n_chunks), dim3(1024), 0, stream, logits, ld, expt_indx, T, E, K, \
                     lay.chunk_tokens, ids, scal, counts)
  if (mode == 0) AF3_TOK(0);
  else if (mode == 1) AF3_TOK(1);
  else AF3_TOK(2);
#undef AF3_TOK
  int rc = af3::check_launch("routing/token_hist");
  if (rc) return rc;
  const int epad = 1 << ebits;  // >= E, <= 1024
  const bool one_scan = lay.rows * epad <= kPlanOneScan;
  if (!one_scan) {
    hipLaunchKernelGGL(plan_prefix_kernel, dim3((unsigned)af3_cdiv(E, kPlanPrefixE)), dim3(1024), 0, stream, counts,
                       n_chunks, E, hist);
    rc = af3::check_launch("routing/prefix");
    if (rc) return rc;
  }
  hipLaunchKernelGGL(plan_scan_kernel, dim3(1), dim3(1024), 0, stream, counts, one_scan ? n_chunks : 0, E, epad, hist,
                     token_offs_raw, m);
  rc = af3::check_launch("routing/scan");
  if (rc) return rc;
  hipLaunchKernelGGL(plan_scatter_kernel, dim3(n_chunks), dim3(256), 0, stream, ids, scal, R, E,
                     lay.chunk_tokens * K, ebits, token_offs_raw, counts, topk_indx, gate_indx, gate_scal);
  return af3::check_launch("routing/scatter");
}

static int routing_common(bool topk, const uint16_t* logits, int64_t ld, const int32_t* expt_indx, int64_t T, int E,
                          int K, uint16_t* gate_scal, int32_t* hist, int32_t* topk_indx, int32_t* gate_indx,
                          int32_t* token_offs_raw, void* workspace, size_t ws_bytes, hipStream_t stream,
                          const PlanMaps* maps = nullptr) {
  AF3_REQUIRE(T >= 0 && E > 0 && K > 0, "routing: bad sizes T=%lld E=%d K=%d", (long long)T, E, K);
  AF3_REQUIRE(K <= 16, "routing: K=%d > 16 unsupported", K);
  AF3_REQUIRE(E <= 0x7fff, "routing: E=%d too large", E);
  AF3_REQUIRE(E * 4 <= 48 * 1024, "routing: E=%d exceeds the per-chunk LDS histogram", E);
  AF3_REQUIRE(!topk || K <= E, "routing: K=%d > E=%d", K, E);
  AF3_REQUIRE(ld >= E, "routing: logits leading dim %lld < E", (long long)ld);
  AF3_REQUIRE(ws_bytes >= (maps ? af3_routing_plan_workspace_bytes(T, E, K, topk)
                                : af3_routing_workspace_bytes(T, E, K)),
              "routing: workspace too small");
  AF3_REQUIRE(!maps || E <= kPlanMaxE, "routing_plan: E=%d above %d", E, kPlanMaxE);
  const int64_t R = T * K;
  AF3_REQUIRE(R < 0x7fffffffLL, "routing: T*K too large");
  char* ws = (char*)workspace;
  const RoutingLayout lay = routing_layout(T, E, K);
  int32_t* ids = (int32_t*)ws;
  uint16_t* scal = (uint16_t*)(ws + lay.scal);
  int32_t* counts = (int32_t*)(ws + lay.counts);
  if (E <= kPlanMaxE) {
    const PlanMaps none{};
    return routing_plan(topk, logits, ld, expt_indx, T, E, K, gate_scal, hist, topk_indx, gate_indx, token_offs_raw,
                        ids, scal, counts, lay, maps ? *maps : none, stream);
  }
  const int n_chunks = (int)lay.rows;

  if (T > 0) {
    dim3 g((unsigned)af3_cdiv(T, 128));
    if (topk)
      hipLaunchKernelGGL(topk_token_kernel, g, dim3(128), 0, stream, logits, ld, T, E, K, ids, scal);
    else
      hipLaunchKernelGGL(replay_token_kernel, g, dim3(128), 0, stream, logits, ld, expt_indx, T, E, K, ids, scal);
    int rc = af3::check_launch("routing/token");
    if (rc) return rc;
    hipLaunchKernelGGL(chunk_hist_kernel, dim3(n_chunks), dim3(kChunk), E * 4, stream, ids, R, E, n_chunks, counts);
    rc = af3::check_launch("routing/hist");
    if (rc) return rc;
    hipLaunchKernelGGL(chunk_scan_kernel, dim3(E), dim3(256), 0, stream, counts, n_chunks, hist);
    rc = af3::check_launch("routing/chunk_scan");
    if (rc) return rc;
  } else {
    hipLaunchKernelGGL(zero_kernel, dim3(1), dim3(256), 0, stream, hist, E);
    int rc = af3::check_launch("routing/zero");
    if (rc) return rc;
  }
  hipLaunchKernelGGL(expert_scan_kernel, dim3(1), dim3(1024), 0, stream, hist, E, token_offs_raw);
  int rc = af3::check_launch("routing/expert_scan");
  if (rc) return rc;
  if (T > 0) {
    hipLaunchKernelGGL(scatter_kernel, dim3(n_chunks), dim3(kChunk), 0, stream, ids, scal, R, n_chunks, token_offs_raw,
                       counts, topk_indx, gate_indx, gate_scal);
    rc = af3::check_launch("routing/scatter");
    if (rc) return rc;
    hipLaunchKernelGGL(fill_tail_kernel, dim3((unsigned)af3_cdiv(R, 256)), dim3(256), 0, stream, token_offs_raw, E,
                       R, topk_indx, gate_scal);
    rc = af3::check_launch("routing/tail");
  }
  return rc;
}

extern "C" int af3_routing_replay(const uint16_t* logits, int64_t ld_logits, const int32_t* expt_indx, int64_t n_tokens,
                                  int n_expts_tot, int n_expts_act, uint16_t* gate_scal, int32_t* hist,
                                  int32_t* topk_indx, int32_t* gate_indx, int32_t* token_offs_raw, void* workspace,
                                  size_t ws_bytes, void* stream) {
  AF3_REQUIRE(expt_indx || n_tokens == 0, "routing_replay: null expt_indx");
  return routing_common(false, logits, ld_logits, expt_indx, n_tokens, n_expts_tot, n_expts_act, gate_scal, hist,
                        topk_indx, gate_indx, token_offs_raw, workspace, ws_bytes, (hipStream_t)stream);
}

// ---- allocation-free routing replay --------------------------------------
// The workspace of af3_routing_replay (ids, softmax weights, per-chunk counts;
// every byte is written before it is read, so nothing needs clearing) lives in
// this file-scope device array.  Each device holds its own copy; host code
// never passes the array's name to a kernel (on the host it only names the
// symbol), it passes the device address taken once per device with
// hipGetSymbolAddress.
constexpr size_t kRoutingScratchBytes = size_t(4) << 20;
static __device__ __align__(256) unsigned char scratch[kRoutingScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

extern "C" size_t af3_routing_scratch_bytes(void) { return kRoutingScratchBytes; }

extern "C" int af3_routing_replay_noalloc(const uint16_t* logits, int64_t ld_logits, const int32_t* expt_indx,
                                          int64_t n_tokens, int n_expts_tot, int n_expts_act, uint16_t* gate_scal,
                                          int32_t* hist, int32_t* topk_indx, int32_t* gate_indx,
                                          int32_t* token_offs_raw, void* stream) {
  AF3_REQUIRE(expt_indx || n_tokens == 0, "routing_replay_noalloc: null expt_indx");
  AF3_REQUIRE(n_tokens >= 0 && n_expts_tot > 0 && n_expts_act > 0, "routing_replay_noalloc: bad sizes");
  const size_t need = af3_routing_workspace_bytes(n_tokens, n_expts_tot, n_expts_act);
  AF3_REQUIRE(need <= kRoutingScratchBytes,
              "routing_replay_noalloc: T=%lld E=%d K=%d needs %zu scratch bytes, the built-in buffer holds %zu "
              "(use af3_routing_replay with a workspace)",
              (long long)n_tokens, n_expts_tot, n_expts_act, need, kRoutingScratchBytes);
  // the array of the device the stream belongs to (the null stream: the
  // current device), taken with that device current
  int cur = 0;
  hipError_t e = hipGetDevice(&cur);
  if (e != hipSuccess) {
    af3::set_error("routing_replay_noalloc: hipGetDevice: %s", hipGetErrorString(e));
    return (int)e;
  }
  hipDevice_t dev = cur;
  if (stream) {
    e = hipStreamGetDevice((hipStream_t)stream, &dev);
    if (e != hipSuccess) {
      af3::set_error("routing_replay_noalloc: hipStreamGetDevice: %s", hipGetErrorString(e));
      return (int)e;
    }
  }
  AF3_REQUIRE(dev >= 0 && dev < kMaxDevices, "routing_replay_noalloc: device %d out of range", (int)dev);
  if (dev != cur && (e = hipSetDevice(dev)) != hipSuccess) {
    af3::set_error("routing_replay_noalloc: hipSetDevice(%d): %s", (int)dev, hipGetErrorString(e));
    return (int)e;
  }
  void* ws = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {  // first call on this device: its copy of the array
      e = hipGetSymbolAddress(&g_scratch_ptr[dev], HIP_SYMBOL(scratch));
      if (e != hipSuccess) g_scratch_ptr[dev] = nullptr;
    }
    ws = g_scratch_ptr[dev];
  }
  int rc = 0;
  if (!ws) {
    af3::set_error("routing_replay_noalloc: hipGetSymbolAddress: %s", hipGetErrorString(e));
    rc = (int)e;
  } else {
    rc = routing_common(false, logits, ld_logits, expt_indx, n_tokens, n_expts_tot, n_expts_act, gate_scal, hist,
                        topk_indx, gate_indx, token_offs_raw, ws, kRoutingScratchBytes, (hipStream_t)stream);
  }
  if (dev != cur) hipSetDevice(cur);  // the caller's current device, as it was
  return rc;
}

extern "C" int af3_routing_topk(const uint16_t* logits, int64_t ld_logits, int64_t n_tokens, int n_expts_tot,
                                int n_expts_act, uint16_t* gate_scal, int32_t* hist, int32_t* topk_indx,
                                int32_t* gate_indx, int32_t* token_offs_raw, void* workspace, size_t ws_bytes,
                                void* stream) {
  return routing_common(true, logits, ld_logits, nullptr, n_tokens, n_expts_tot, n_expts_act, gate_scal, hist,
                        topk_indx, gate_indx, token_offs_raw, workspace, ws_bytes, (hipStream_t)stream);
}

extern "C" size_t af3_routing_plan_workspace_bytes(int64_t n_tokens, int n_expts_tot, int n_expts_act, int topk) {
  if (plan_one_block(topk != 0, n_tokens, n_expts_tot, n_expts_act) && !(topk && n_expts_tot > kPlanMaxTopkE)) return 0;
  return af3_routing_workspace_bytes(n_tokens, n_expts_tot, n_expts_act);
}

// Routing and the grouped GEMM's tile metadata in one call (af3_routing_replay
// / af3_routing_topk, then af3_expt_data and af3_tile_order per block size).
extern "C" int af3_routing_plan(const uint16_t* logits, int64_t ld_logits, const int32_t* expt_indx, int topk,
                                int64_t n_tokens, int n_expts_tot, int n_expts_act, uint16_t* gate_scal, int32_t* hist,
                                int32_t* topk_indx, int32_t* gate_indx, int32_t* token_offs_raw, const int32_t* block_ms,
                                int n_block_ms, int n_orders, int max_tiles, int32_t* token_offs_pad,
                                int32_t* block_pid_map, int32_t* orders, void* workspace, size_t ws_bytes,
                                void* stream) {
  AF3_REQUIRE(block_ms && n_block_ms > 0 && n_block_ms <= kPlanMaxBm && n_orders >= 0 && n_orders <= n_block_ms &&
                  max_tiles >= 0,
              "routing_plan: bad block sizes (%d, %d orders, max_tiles %d)", n_block_ms, n_orders, max_tiles);
  AF3_REQUIRE(n_expts_tot <= kPlanMaxE, "routing_plan: E=%d above %d", n_expts_tot, kPlanMaxE);
  AF3_REQUIRE(token_offs_pad && (max_tiles == 0 || (block_pid_map && (n_orders == 0 || orders))),
              "routing_plan: null pointer");
  PlanMaps m{};
  m.n_bm = n_block_ms;
  m.n_order = n_orders;
  m.max_tiles = max_tiles;
  for (int i = 0; i < n_block_ms; ++i) {
    AF3_REQUIRE(block_ms[i] > 0, "routing_plan: block size %d", block_ms[i]);
    m.bm[i] = block_ms[i];
  }
  m.offs_pad = token_offs_pad;
  m.map = block_pid_map;
  m.order = orders;
  AF3_REQUIRE(topk || expt_indx || n_tokens == 0, "routing_plan: null expt_indx");
  return routing_common(topk != 0, logits, ld_logits, expt_indx, n_tokens, n_expts_tot, n_expts_act,
                        gate_scal, hist, topk_indx, gate_indx, token_offs_raw, workspace, ws_bytes,
                        (hipStream_t)stream, &m);
}

extern "C" int af3_expt_data(const int32_t* hist, int n_expts_tot, const int32_t* block_ms_dev, int n_block_ms,
                             int max_tiles, int32_t* token_offs_pad, int32_t* block_pid_map, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  AF3_REQUIRE(n_expts_tot > 0 && n_expts_tot <= kScanMaxE && n_block_ms > 0 && n_block_ms <= 64 && max_tiles >= 0,
              "expt_data: bad sizes (E=%d, block sizes %d, max_tiles %d)", n_expts_tot, n_block_ms, max_tiles);
  hipLaunchKernelGGL(tile_scan_map_kernel, dim3(n_block_ms), dim3(1024), 0, stream, hist, n_expts_tot, block_ms_dev,
                     max_tiles, token_offs_pad, block_pid_map);
  return af3::check_launch("expt_data");
}

// Order of the BM-row tiles for the grouped GEMM's work list (same entries as
// the block_pid_map of af3_expt_data for this BM, permuted): full tiles in
// expert order, then each expert's partial last tile by decreasing rows.
extern "C" int af3_tile_order(const int32_t* hist, int n_expts_tot, int block_m, const int32_t* token_offs_pad,
                              int max_tiles, int32_t* order, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  AF3_REQUIRE(n_expts_tot > 0 && n_expts_tot <= kSchedMaxE, "tile_order: E=%d outside [1, %d]", n_expts_tot,
              kSchedMaxE);
  AF3_REQUIRE(block_m > 0 && block_m <= kSchedMaxBM && max_tiles >= 0, "tile_order: bad block_m %d / max_tiles %d",
              block_m, max_tiles);
  AF3_REQUIRE(max_tiles == 0 || (hist && token_offs_pad && order), "tile_order: null pointer");
  if (max_tiles == 0) return 0;
  (void)token_offs_pad;  // the kernel counts the tiles itself (the same total as token_offs_pad[E])
  hipLaunchKernelGGL(tile_order_kernel, dim3(1), dim3(1024), 0, stream, hist, n_expts_tot, block_m, max_tiles, order);
  return af3::check_launch("tile_order");
}
