// Expert-LoRA merge for weight sync: one bf16 weight per expert with the
// adapter folded in,
//
//   W'[e][n][k] = bf16( float(deq(W[e])[n][k]) + s * sum_j B[e][n][j] * A[e][j][k] )
//
// deq = the MXFP4 -> bf16 rule of the dequant kernel (kernels.py:120-158),
// A [E][r][K] and B [E][N][r] bf16 (the adapter layout of the experts module),
// s = lora_alpha / r.  The arithmetic follows the reference's LoRA merge for
// sglang sync (model_trainer.py:653-719, arithmetic at 710-712): base and delta in fp32, the product
// B @ A scaled after the sum, one rounding to bf16 (round to nearest even).
//
// Output layouts: 0 = [E][N][K] (the frozen weight's own row order),
// 1 = [E][K][N] (transformers' GptOssExperts parameter, modeling_gpt_oss.py:75-77,
// the layout a bf16 gpt-oss checkpoint holds).
//
// Ranks above 64 take the general kernel: a tile = 64(n) x 64(k) of one expert,
// persistent blocks of 4 waves walk the tiles.  The rank-r delta runs on
// v_mfma_f32_32x32x16_bf16 (products of bf16 are exact in fp32), each wave one
// 32x32 sub-tile (A's k-slice staged in LDS with 16-byte loads), the result
// staged in LDS as fp32.  Then each thread dequantises a quarter MXFP4 block (8
// values) of two rows, adds the delta and writes 16 B of bf16 per row: straight to
// HBM for layout 0, through an LDS transpose for layout 1 (64-column runs of 128
// B, whole lines per store).  HBM-bound: per output element 2 B written and 17/32
// B of packed weight read; the adapters are re-read from L2.
#include <type_traits>

#include "af3_common.h"

namespace {

constexpr int kMgN = 64;
constexpr int kMgK = 64;
constexpr int kMgDP = 68;  // fp32 pitch of the delta tile (16-lane groups of the row reads hit distinct banks)
constexpr int kMgMP = 66;  // u16 pitch of the merged tile (transposed reads hit distinct banks)
constexpr int kMgLP = 72;  // u16 pitch of the staged A slice (16-byte rows; the half-waves' rows 32 banks apart)
static_assert(kMgN * kMgMP <= kMgN * kMgLP, "merged tile must fit the staging buffer");
constexpr int kMgBlocksPerXcd = 32 * 6;

struct MergeTile {
  int e, n0, k0;
};

__device__ __forceinline__ MergeTile merge_tile(int64_t tile, int n_tiles_n, int n_tiles_k) {
  const int64_t rest = tile / n_tiles_k;
  return {(int)(rest / n_tiles_n), (int)(rest % n_tiles_n) * kMgN, (int)(tile % n_tiles_k) * kMgK};
}

// The packed dword (8 consecutive k) of rows p*32 + tid/8, p = 0, 1, of a tile.
__device__ __forceinline__ void merge_load_packed(const uint8_t* __restrict__ blocks,
                                                  const uint8_t* __restrict__ scales, MergeTile t, int N, int K,
                                                  int tid, uint32_t v[2], uint32_t sc[2]) {
  const int k = t.k0 + (tid & 7) * 8;
  const int G = K >> 5;
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int n = t.n0 + p * 32 + (tid >> 3);
    v[p] = 0u;
    sc[p] = 0u;
    if (n < N && k < K) {
      const int64_t grp = ((int64_t)t.e * N + n) * G + (k >> 5);
      v[p] = __builtin_nontemporal_load((const uint32_t*)(blocks + grp * 16 + ((k & 31) >> 1)));
      sc[p] = scales[grp];
    }
  }
}

// Persistent blocks: block b serves XCD b % 8 and walks that XCD's contiguous run of
// tiles (k fastest) with stride blocks_per_xcd, so the neighbouring k-tiles of a row,
// which share lines of the packed weight and its scales, are in flight together in one
// L2.  The next tile's packed dwords are loaded while the current tile is computed.
__global__ __launch_bounds__(256, 6) void lora_merge_generic_kernel(const uint8_t* __restrict__ blocks,
                                                         const uint8_t* __restrict__ scales,
                                                         const uint16_t* __restrict__ la,
                                                         const uint16_t* __restrict__ lb, float s,
                                                         uint16_t* __restrict__ out, int N, int K, int r,
                                                         int layout, int n_tiles_n, int n_tiles_k, int64_t n_tiles,
                                                         int64_t per_xcd, int blocks_per_xcd) {
  __shared__ __attribute__((aligned(16))) float D[kMgN * kMgDP];
  // A's k-slice (up to 64 of its r rows at a time) before the MFMA, the merged tile after it
  __shared__ __attribute__((aligned(16))) uint16_t LM[kMgN * kMgLP];
  uint16_t* const La = LM;
  uint16_t* const Mt = LM;
  const int tid = threadIdx.x;
  const int w = tid >> 6;
  const int lane = tid & 63;
  const int xcd = blockIdx.x & 7;
  const int64_t t_end = min(n_tiles, (int64_t)(xcd + 1) * per_xcd);
  int64_t tile = (int64_t)xcd * per_xcd + (blockIdx.x >> 3);
  uint32_t v[2] = {0u, 0u}, sc[2] = {0u, 0u};
  if (tile < t_end) merge_load_packed(blocks, scales, merge_tile(tile, n_tiles_n, n_tiles_k), N, K, tid, v, sc);

  for (; tile < t_end; tile += blocks_per_xcd) {
    const MergeTile t = merge_tile(tile, n_tiles_n, n_tiles_k);
    const int e = t.e, n0 = t.n0, k0 = t.k0;
    uint32_t vn[2] = {0u, 0u}, scn[2] = {0u, 0u};
    if (tile + blocks_per_xcd < t_end)
      merge_load_packed(blocks, scales, merge_tile(tile + blocks_per_xcd, n_tiles_n, n_tiles_k), N, K, tid, vn, scn);

    // ---- delta = B[e][n0.., :] @ A[e][:, k0..] on the MFMA, one 32x32 sub-tile per wave
    {
      const int nr = n0 + (w >> 1) * 32 + (lane & 31);
      const int kcl = (w & 1) * 32 + (lane & 31);
      af3_f32x16 acc;
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = 0.f;
      for (int jc = 0; jc < r; jc += 64) {
        // stage A[e][jc .. jc+64)[k0 .. k0+64) in LDS with 16-byte loads (the MFMA wants
        // 8 consecutive j per lane, which run down A's columns); the barrier also ends
        // the previous tile's reads of the merged tile that shares this buffer
        const int rc = min(64, r - jc);
        __syncthreads();
        for (int j = tid >> 3; j < rc; j += 32) {
          const int kk = k0 + (tid & 7) * 8;
          af3_u32x4 val = {0u, 0u, 0u, 0u};
          if (kk < K) val = *(const af3_u32x4*)(la + ((int64_t)e * r + jc + j) * K + kk);
          *(af3_u32x4*)(La + j * kMgLP + (tid & 7) * 8) = val;
        }
        __syncthreads();
        for (int j0 = 0; j0 < rc; j0 += 16) {
          const int jl = j0 + (lane >> 5) * 8;  // this lane's 8 reduction indices (r % 8 == 0)
          af3_u32x4 aw = {0u, 0u, 0u, 0u};
          uint32_t bw[4] = {0u, 0u, 0u, 0u};
          if (jl < rc) {
            if (nr < N) aw = *(const af3_u32x4*)(lb + ((int64_t)e * N + nr) * r + jc + jl);
#pragma unroll
            for (int q = 0; q < 4; ++q)
              bw[q] = (uint32_t)La[(jl + 2 * q) * kMgLP + kcl] | ((uint32_t)La[(jl + 2 * q + 1) * kMgLP + kcl] << 16);
          }
          const af3_bf16x8 a = __builtin_bit_cast(af3_bf16x8, aw);
          const af3_bf16x8 b = __builtin_bit_cast(af3_bf16x8, (af3_u32x4){bw[0], bw[1], bw[2], bw[3]});
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
        }
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = (w >> 1) * 32 + (i >> 2) * 8 + (lane >> 5) * 4 + (i & 3);
        D[row * kMgDP + kcl] = acc[i] * s;
      }
    }
    __syncthreads();

    // ---- dequantise + add; thread = 8 consecutive k of rows p*32 + tid/8 (eight lanes
    // span a 128-byte output run, so each 16-byte store instruction writes whole lines)
    const int kl = (tid & 7) * 8;
    const int k = k0 + kl;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int nl = p * 32 + (tid >> 3);
      const bool live = n0 + nl < N && k < K;
      uint32_t m[4] = {0u, 0u, 0u, 0u};
      if (live) {
        uint32_t q[4];
        af3_dequant_u32(v[p], sc[p], q);
        const float4* d4 = (const float4*)(D + nl * kMgDP + kl);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const float4 d = d4[c];
          const uint32_t lo = q[2 * c], hi = q[2 * c + 1];
          m[2 * c] = af3_pack_bf16x2(af3_bf16_to_f32(lo & 0xFFFFu) + d.x, af3_bf16_to_f32(lo >> 16) + d.y);
          m[2 * c + 1] = af3_pack_bf16x2(af3_bf16_to_f32(hi & 0xFFFFu) + d.z, af3_bf16_to_f32(hi >> 16) + d.w);
        }
      }
      if (layout == 0) {
        if (live)
          __builtin_nontemporal_store((af3_u32x4){m[0], m[1], m[2], m[3]},
                                      (af3_u32x4*)(out + ((int64_t)e * N + n0 + nl) * K + k));
      } else {
        uint32_t* mrow = (uint32_t*)(Mt + nl * kMgMP + kl);
#pragma unroll
        for (int c = 0; c < 4; ++c) mrow[c] = m[c];
      }
    }

    if (layout != 0) {
      // ---- layout 1: transposed through LDS; thread = 8 consecutive n of k row p*32 + tid/8
      __syncthreads();
      const int nt = (tid & 7) * 8;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int kt = p * 32 + (tid >> 3);
        const int kk = k0 + kt;
        if (kk >= K) break;
        uint32_t t4[4];
#pragma unroll
        for (int c = 0; c < 4; ++c)
          t4[c] = (uint32_t)Mt[(nt + 2 * c) * kMgMP + kt] | ((uint32_t)Mt[(nt + 2 * c + 1) * kMgMP + kt] << 16);
        uint16_t* o = out + ((int64_t)e * K + kk) * N + n0 + nt;
        if ((N & 7) == 0 && n0 + nt + 8 <= N) {
          __builtin_nontemporal_store((af3_u32x4){t4[0], t4[1], t4[2], t4[3]}, (af3_u32x4*)o);
        } else {
          for (int c = 0; c < 8 && n0 + nt + c < N; ++c) o[c] = (uint16_t)(t4[c >> 1] >> (16 * (c & 1)));
        }
      }
    }
    v[0] = vn[0];
    v[1] = vn[1];
    sc[0] = scn[0];
    sc[1] = scn[1];
  }
}

// The merge for r <= 64: a unit is one (expert, 256-column k-tile, run of 64-row
// n-tiles), and each of the block's eight waves walks the run on its own, with no
// block barrier: LAYOUT 1 [E][K][N] takes 64 n x 32 k per wave and tile, LAYOUT 0
// [E][N][K] 32 n x 64 k.  The rows of the MFMA's A operand (the adapter's k
// columns) are permuted so that the 16 accumulators of a lane are 16 consecutive
// k of one n: its packed codes are one run of 8 bytes, dequantised and summed in
// registers, and only the bf16 result goes through LDS (wave-private), once, to
// turn it into 128-byte output runs.  The A fragments stay in registers along the
// run; the next tile's codes, scales and B fragments are loaded while the current
// tile is computed.
// HBM bounds it, and the reads cost more than their share: 32 experts' gate_up at
// r 16 take 159 us [E][K][N] / 112 us [E][N][K] without the stores, and 251 / 200
// us with loads that all hit in L2, where the whole takes 362 / 337.  So a unit
// reads 128 bytes of each packed row (a whole line; 64 bytes per unit: 387 / 343
// us, codes loaded non-temporally: 517 / 344), and units are dealt to the XCDs
// in contiguous runs (k-tile fastest), so the blocks that share lines of packed
// rows and scales run on one L2.  Runs of 8 n-tiles: 16 381 / 341, 4 367 / 321 at
// r 16 but no better at r 32.  Two to six tiles of loads in flight changed
// nothing.  Against the form before (64 x 64 tiles by four waves together, the
// delta as fp32 and the sum as bf16 through LDS, three block barriers per tile):
// r 16 377 / 370 -> 362 / 337 us (1.36 GB, 3.7 / 4.0 TB/s), r 32 411 / 405 -> 409 /
// 352, r 64 538 / 532 -> 525 / 447.
constexpr int kMgWaves = 8;     // waves of a block
constexpr int kMgBK = 32 * kMgWaves;  // k columns of a unit
constexpr int kMgRun = 8;       // n-tiles of a unit (fewer where the launch has few units)
constexpr int kMgTP = 72;       // u16 pitch of a wave's result tile (16-byte rows)
constexpr int kMgUnits = 1024;  // units below which the runs are halved
typedef af3_u32x4 mg_u32x4_a4 __attribute__((aligned(4)));  // the packed blocks are 4-byte aligned
typedef __attribute__((ext_vector_type(2))) uint32_t mg_u32x2;
typedef mg_u32x2 mg_u32x2_a4 __attribute__((aligned(4)));

__device__ __forceinline__ void mg_wave_sync() {  // orders a wave's LDS accesses (the LDS keeps their order)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// RQ: 16-deep MFMA steps of the rank
template <int LAYOUT, int RQ>
__global__ __launch_bounds__(64 * kMgWaves, RQ <= 2 ? 4 : 2) void lora_merge_kernel(
    const uint8_t* __restrict__ blocks, const uint8_t* __restrict__ scales, const uint16_t* __restrict__ la,
    const uint16_t* __restrict__ lb, float s, uint16_t* __restrict__ out, int N, int K, int r, int n_tiles_n,
    int n_tiles_k, int run_tiles, int n_runs, int n_units, int per_xcd) {
#pragma clang fp contract(off)
  constexpr int NT = LAYOUT ? 2 : 1, KT = LAYOUT ? 1 : 2;  // 32-wide sub-tiles of a wave along n and k
  __shared__ __attribute__((aligned(16))) uint16_t lds[kMgWaves][32 * kMgTP];
  const int unit = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if (unit >= n_units || unit >= ((int)(blockIdx.x & 7) + 1) * per_xcd) return;
  const int rest = unit / n_tiles_k;
  const int e = rest / n_runs;
  const int t_first = (rest % n_runs) * run_tiles;
  const int t_last = min(n_tiles_n, t_first + run_tiles);
  const int G = K >> 5;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 31, h = lane >> 5;
  const int kw = (unit % n_tiles_k) * kMgBK + (LAYOUT ? w * 32 : (w % (kMgWaves / 2)) * 64);  // the wave's first k
  const int nw = LAYOUT ? 0 : (w / (kMgWaves / 2)) * 32;  // its first n in a tile
  if (kw >= K) return;
  uint16_t* const T = lds[w];

  // A operand: MFMA row m = 8 j + 4 h + q is k = kw + (LAYOUT 1: 16, else 32) h + 16 t + 4 j + q
  af3_bf16x8 af[KT][RQ];
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    const int k = kw + ((c >> 2) & 1) * (LAYOUT ? 16 : 32) + t * 16 + 4 * (c >> 3) + (c & 3);
    const uint16_t* a_k = la + (int64_t)e * r * K + min(k, K - 1);  // columns past K are not stored
#pragma unroll
    for (int q = 0; q < RQ; ++q) {
      const int j = q * 16 + h * 8;  // 8 reduction indices (r % 8 == 0)
      uint32_t v[4] = {0u, 0u, 0u, 0u};
      if (j < r)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          v[i] = (uint32_t)a_k[(int64_t)(j + 2 * i) * K] | ((uint32_t)a_k[(int64_t)(j + 2 * i + 1) * K] << 16);
      af[t][q] = __builtin_bit_cast(af3_bf16x8, (af3_u32x4){v[0], v[1], v[2], v[3]});
    }
  }

  // a lane's codes: LAYOUT 1 half a block (16 k) of rows c and 32 + c, else the block (32 k) of row c
  const int kb = min((kw >> 5) + (LAYOUT ? 0 : h), G - 1);
  struct Tile {
    uint32_t v[4], sc[NT];
    af3_u32x4 b[NT][RQ];
  };
  auto fetch = [&](int ti, Tile& d) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int64_t row = (int64_t)e * N + min(ti * kMgN + nw + t * 32 + c, N - 1);  // rows past N are not stored
      const int64_t grp = row * G + kb;
      if constexpr (LAYOUT) {
        const mg_u32x2 x = *(const mg_u32x2_a4*)(blocks + grp * 16 + h * 8);
        d.v[2 * t] = x[0];
        d.v[2 * t + 1] = x[1];
      } else {
        const af3_u32x4 x = *(const mg_u32x4_a4*)(blocks + grp * 16);
#pragma unroll
        for (int i = 0; i < 4; ++i) d.v[i] = x[i];
      }
      d.sc[t] = scales[grp];
#pragma unroll
      for (int q = 0; q < RQ; ++q)  // no branch: lanes past the rank load its last indices and zero them before use
        d.b[t][q] = *(const af3_u32x4*)(lb + row * r + min(q * 16 + h * 8, r - 8));
    }
  };
  const bool tail_rank = r < RQ * 16;
  // one tile from `cur`, the next one's operands into `nxt`. WHOLE: every store
  // unconditional, so that the compiler's wait for `nxt` counts them and leaves
  // them in flight
  auto step = [&](auto whole_c, int ti, Tile& cur, Tile& nxt) {
    constexpr bool WHOLE = decltype(whole_c)::value;
    const int n0 = ti * kMgN;
    fetch(min(ti + 1, t_last - 1), nxt);
    if (tail_rank) {
#pragma unroll
      for (int q = 0; q < RQ; ++q)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) cur.b[t][q][i] = q * 16 + h * 8 < r ? cur.b[t][q][i] : 0u;
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {  // the two 32 x 32 sub-tiles
      af3_f32x16 acc;
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
      for (int q = 0; q < RQ; ++q)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[LAYOUT ? 0 : u][q],
                                                      __builtin_bit_cast(af3_bf16x8, cur.b[LAYOUT ? u : 0][q]), acc, 0,
                                                      0, 0);
      uint32_t m[8];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        uint32_t d[4];
        af3_dequant_u32(cur.v[2 * u + p], cur.sc[LAYOUT ? u : 0], d);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float lo = acc[8 * p + 2 * i] * s, hi = acc[8 * p + 2 * i + 1] * s;
          m[4 * p + i] = af3_pack_bf16x2(af3_bf16_to_f32(d[i] & 0xFFFFu) + lo, af3_bf16_to_f32(d[i] >> 16) + hi);
        }
      }
      if constexpr (LAYOUT) {  // T[k][n]
        uint16_t* const col = T + h * 16 * kMgTP + u * 32 + c;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          col[2 * i * kMgTP] = (uint16_t)m[i];
          col[(2 * i + 1) * kMgTP] = (uint16_t)(m[i] >> 16);
        }
      } else {  // T[n][k]
        af3_u32x4* const row = (af3_u32x4*)(T + c * kMgTP + h * 32 + u * 16);
        row[0] = (af3_u32x4){m[0], m[1], m[2], m[3]};
        row[1] = (af3_u32x4){m[4], m[5], m[6], m[7]};
      }
    }
    mg_wave_sync();
    const int tr = lane >> 3, tc = (lane & 7) * 8;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int rr = i * 8 + tr;
      const af3_u32x4 v = *(const af3_u32x4*)(T + rr * kMgTP + tc);
      if constexpr (LAYOUT) {
        uint16_t* const o = out + ((int64_t)e * K + kw + rr) * N + n0 + tc;
        if (WHOLE || (N & 7) == 0) {
          if (WHOLE || n0 + tc < N) __builtin_nontemporal_store(v, (af3_u32x4*)o);
        } else {
          for (int x = 0; x < 8; ++x)
            if (n0 + tc + x < N) o[x] = (uint16_t)(v[x >> 1] >> (16 * (x & 1)));
        }
      } else {
        const int n = n0 + nw + rr;
        if (WHOLE || (n < N && kw + tc < K))
          __builtin_nontemporal_store(v, (af3_u32x4*)(out + ((int64_t)e * N + n) * K + kw + tc));
      }
    }
    mg_wave_sync();
  };
  auto walk = [&](auto whole_c) {
    Tile a, b;
    fetch(t_first, a);
    for (int ti = t_first;;) {
      step(whole_c, ti, a, b);
      if (++ti >= t_last) break;
      step(whole_c, ti, b, a);
      if (++ti >= t_last) break;
    }
  };
  if (t_last * kMgN <= N && (LAYOUT ? (N & 7) == 0 : kw + 64 <= K))
    walk(std::true_type{});
  else
    walk(std::false_type{});
}

}  // namespace

extern "C" int af3_mxfp4_lora_merge(const uint8_t* blocks, const uint8_t* scales, const uint16_t* lora_a,
                                    const uint16_t* lora_b, float scaling, uint16_t* out, int E, int N, int K, int r,
                                    int layout, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  AF3_REQUIRE(E >= 0 && N >= 0 && K >= 0 && E <= 65535, "mxfp4_lora_merge: bad sizes");
  AF3_REQUIRE(K % 32 == 0, "mxfp4_lora_merge: K must be a multiple of 32 (one MXFP4 block)");
  AF3_REQUIRE(r > 0 && r % 8 == 0 && r <= 256, "mxfp4_lora_merge: rank must be a positive multiple of 8, <= 256");
  AF3_REQUIRE(layout == 0 || layout == 1, "mxfp4_lora_merge: layout must be 0 ([E,N,K]) or 1 ([E,K,N])");
  if ((int64_t)E * N * K == 0) return 0;
  AF3_REQUIRE(blocks && scales && lora_a && lora_b && out, "mxfp4_lora_merge: null pointer");
  AF3_REQUIRE(((uintptr_t)blocks & 3) == 0 && ((uintptr_t)lora_b & 15) == 0 && ((uintptr_t)lora_a & 15) == 0 &&
                  ((uintptr_t)out & 15) == 0,
              "mxfp4_lora_merge: blocks must be 4-byte, lora_a, lora_b and out 16-byte aligned");
  const int ntn = (int)af3_cdiv(N, kMgN);
  if (r <= 64) {
    const int nk = (int)af3_cdiv(K, kMgBK);
    int run = kMgRun;  // shorter runs while the launch would leave CUs idle
    while (run > 2 && (int64_t)E * af3_cdiv(ntn, run) * nk < kMgUnits) run /= 2;
    const int runs = (int)af3_cdiv(ntn, run);
    const int64_t units = (int64_t)E * runs * nk;
    AF3_REQUIRE(units <= 0x7ffffff0LL && (int64_t)kMgN * N <= 0x7fffffffLL && (int64_t)kMgK * N <= 0x7fffffffLL,
                "mxfp4_lora_merge: tensor too large");
    const int upx = (int)af3_cdiv(units, 8);
#define AF3_MG(lay, rq)                                                                                        \
  hipLaunchKernelGGL((lora_merge_kernel<lay, rq>), dim3((unsigned)(8 * upx)), dim3(64 * kMgWaves), 0, stream,  \
                     blocks, scales, lora_a, lora_b, scaling, out, N, K, r, ntn, nk, run, runs, (int)units, upx)
#define AF3_MGR(lay)              \
  do {                            \
    if (r <= 16) AF3_MG(lay, 1);  \
    else if (r <= 32) AF3_MG(lay, 2); \
    else AF3_MG(lay, 4);          \
  } while (0)
    if (layout) AF3_MGR(1);
    else AF3_MGR(0);
#undef AF3_MGR
#undef AF3_MG
  } else {
    const int ntk = (int)af3_cdiv(K, kMgK);
    const int64_t tiles = (int64_t)E * ntn * ntk;
    const int64_t per_xcd = af3_cdiv(tiles, 8);
    // resident blocks per XCD: 32 CUs x 6 blocks of 26 KB LDS
    const int bpx = (int)(per_xcd < kMgBlocksPerXcd ? per_xcd : kMgBlocksPerXcd);
    hipLaunchKernelGGL(lora_merge_generic_kernel, dim3((unsigned)(8 * bpx)), dim3(256), 0, stream, blocks, scales,
                       lora_a, lora_b, scaling, out, N, K, r, layout, ntn, ntk, tiles, per_xcd, bpx);
  }
  return af3::check_launch("mxfp4_lora_merge");
}
