// Router logits of the gpt-oss MoE layer on bf16 MFMA.
//
// Reference behaviour (quantization.py:653-654, mlp_forward):
//   router_logits = nn.functional.linear(hidden_states, router.weight, router.bias)
// i.e. logits[t][e] = bf16(sum_k x[t][k] W[e][k] + b[e]) with fp32 sums, for
// hidden_states [T, H] bf16, W [E, H] bf16, b [E] bf16.  The logits then feed
// the top-k / replay routing (routing.hip).
//
// The product is skinny (E = 32 or 128 columns): a block takes 64 rows by all
// E columns, its waves one 32 x 32 (E > 128: 32 x 64) tile each, and walks k in
// 64-deep steps.  With one block per CU (16384 rows) or fewer nothing hides a
// k-step's load latency, and that latency times H / 64 steps is what a plain
// double buffer costs whatever the row count (33-53 us, 1 row or 16384, where
// the x read of 16384 rows takes 15 us).  So the x rows ([64][64] bf16) and
// the W tile ([E][64]) of a k-step go global -> LDS through a ring of kRtStages
// stages, all but one of them in flight, one barrier per step; the sums keep
// their order, so the logits are unchanged.  Measured: 1
// row, E 128 36 -> 16 us; 23 rows, E 32 33 -> 14; 4096 rows, E 32 41 -> 18; 1021
// rows, E 128 48 -> 24; 16384 rows, E 128 53 -> 30 (LDS reads bound it now).
// Several blocks per CU hide each other's latency, and what the ring's depth costs
// is blocks per CU: past 256 blocks it has two stages (three at E 65 - 128 and H
// >= 2048, where the W tile's latency shows), and 129 - 192 experts are padded to
// 192 columns instead of 256 where the products count (H >= 512).  65536 rows,
// kernel time, plain double buffer / deep ring / these: H 2880, E 8 64 / 66 / 64,
// E 128 114 / 104 / 100, E 160 125 / 136 / 116, E 256 167 / 149 / 139; H 512, E 64
// 15 / 22 / 14, E 128 20 / 27 / 17; H 64, E 128 8.7 / 12.8 / 7.5.
// LDS chunks of 16 bytes are XOR-swizzled by row (the copy writes LDS linearly,
// so the lanes' source addresses carry the swizzle).  k is permuted
// identically on both operands: lane (r, h) of v_mfma_f32_32x32x16_bf16 feeds
// k = 32 h + 8 s + (0..7) at sub-step s.
#include "af3_common.h"

namespace {

constexpr int kRtRows = 64;  // rows per block
constexpr int kRtBK = 64;    // k per step
constexpr unsigned kRtOneRound = 256;  // blocks up to which the deep rings are taken (one per CU)

// one 16-byte global -> LDS copy per lane (LDS address: wave-uniform base + 16 lane)
__device__ __forceinline__ void rt_dma16(const void* gptr, uint32_t lds_byte_addr) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(gptr), "{m0}"(lds_byte_addr) : "memory");
}

// EP columns computed (E rounded up to 32, 64, 128, 192 or 256), TW 32-column tiles per wave, ST ring stages
// (ONCE: no k-step is copied twice, two stages only)
template <int EP, int TW, int ST, bool ONCE = false>
__global__ __launch_bounds__(EP / TW * 4) void router_kernel(const uint16_t* __restrict__ x, int64_t ldx,
                                                             const uint16_t* __restrict__ w, int64_t ldw,
                                                             const uint16_t* __restrict__ bias, int64_t T, int H, int E,
                                                             uint16_t* __restrict__ out, int64_t ldo) {
  constexpr int NW = EP / TW / 16;                 // waves: 2 row groups x EP / (32 TW) column groups
  constexpr int STAGE = (kRtRows + EP) * 128;      // bytes: x rows, then W rows
  constexpr int CPW = (kRtRows + EP) / 8 / NW;     // 1 KB copies (8 rows) per wave and k-step
  static_assert((kRtRows + EP) / 8 % NW == 0, "whole copies per wave");
  static_assert(CPW * (ST - 2) <= 31 && ST * STAGE <= 160 * 1024, "ring");
  __shared__ __attribute__((aligned(16))) uint8_t lds[ST * STAGE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 31, lh = lane >> 5;
  const int rg = wave & 1, cg = wave >> 1;
  const int nk = H / kRtBK;
  const int64_t row0 = (int64_t)blockIdx.x * kRtRows;
  const bool rows = row0 + rg * 32 < T;  // else the wave only copies and keeps the barriers

  // copy j of the wave: rows 8 (wave CPW + j) .. + 7 of the stage, lane l row l / 8, 16-byte slot l % 8
  const uint16_t* src[CPW];
#pragma unroll
  for (int j = 0; j < CPW; ++j) {
    const int r = (wave * CPW + j) * 8 + (lane >> 3);
    const int ch = (lane & 7) ^ (r & 7);
    if (r < kRtRows)  // rows past T: any valid row (their results are not stored)
      src[j] = x + min(row0 + r, T - 1) * ldx + ch * 8;
    else
      src[j] = w + (int64_t)min(r - kRtRows, E - 1) * ldw + ch * 8;
  }
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)lds);
  // k-steps past the end copy the last one again, into a stage no wave reads again (no branch
  // in the loop), unless there are so few that this counts
  static_assert(!ONCE || ST == 2, "the wait counts the repeated copies");
  auto issue = [&](int kk) {
    if (ONCE && kk >= nk) return;
    const int ks = min(kk, nk - 1);
    const uint32_t st = lds0 + (uint32_t)((kk % ST) * STAGE + wave * CPW * 1024);
#pragma unroll
    for (int j = 0; j < CPW; ++j) rt_dma16(src[j] + ks * kRtBK, st + (uint32_t)(j * 1024));
  };

  af3_f32x16 acc[TW];
#pragma unroll
  for (int t = 0; t < TW; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;

#pragma unroll
  for (int k = 0; k < ST - 1; ++k) issue(k);
  for (int kk = 0; kk < nk; ++kk) {
    // this wave's copies of k-step kk have landed (those of the ST - 2 newer
    // steps may be outstanding); then the barrier: every wave's have, and every
    // wave has read stage kk - 1, which the next copies overwrite
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(CPW * (ST - 2)) : "memory");
    issue(kk + ST - 1);
    if (!rows) continue;
    const uint8_t* const st = lds + (kk % ST) * STAGE;
    const uint8_t* const ar = st + (rg * 32 + lr) * 128;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int ch = ((lh * 4 + s) ^ (lr & 7)) << 4;
      const af3_bf16x8 a = *(const af3_bf16x8*)(ar + ch);
#pragma unroll
      for (int t = 0; t < TW; ++t) {
        const af3_bf16x8 b = *(const af3_bf16x8*)(st + (kRtRows + (cg * TW + t) * 32 + lr) * 128 + ch);
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[t], 0, 0, 0);
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the repeated last copies, before the LDS is given back
  // epilogue: lane (c, h) of sub-tile t holds rows 8 j + 4 h + q, column 32 (cg TW + t) + c
#pragma unroll
  for (int t = 0; t < TW; ++t) {
    const int col = (cg * TW + t) * 32 + lr;
    if (col >= E) continue;
    const float b = bias ? af3_bf16_to_f32(bias[col]) : 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t r = row0 + rg * 32 + 8 * j + 4 * lh + q;
        if (r < T) out[r * ldo + col] = (uint16_t)af3_f32_to_bf16(acc[t][4 * j + q] + b);
      }
  }
}

template <int EP, int TW, int ST, bool ONCE = false>
constexpr unsigned router_threads() {
  return EP / TW * 4;
}

}  // namespace

extern "C" int af3_router_logits(const uint16_t* x, int64_t ldx, const uint16_t* w, int64_t ldw, const uint16_t* bias,
                                 int64_t n_tokens, int hidden, int n_expts, uint16_t* logits, int64_t ld_logits,
                                 void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  AF3_REQUIRE(n_tokens >= 0 && hidden > 0 && n_expts > 0, "router_logits: bad sizes");
  AF3_REQUIRE(n_expts <= 256, "router_logits: E=%d above 256", n_expts);
  AF3_REQUIRE(hidden % kRtBK == 0, "router_logits: hidden size %d must be a multiple of %d", hidden, kRtBK);
  AF3_REQUIRE(ldx >= hidden && ldw >= hidden && ld_logits >= n_expts, "router_logits: bad leading dimensions");
  AF3_REQUIRE(ldx % 8 == 0 && ldw % 8 == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0,
              "router_logits: x and W rows must be 16-byte aligned");
  if (n_tokens == 0) return 0;
  AF3_REQUIRE(x && w && logits, "router_logits: null pointer");
  const dim3 grid((unsigned)af3_cdiv(n_tokens, kRtRows));
#define AF3_RT(...)                                                                                               \
  hipLaunchKernelGGL((router_kernel<__VA_ARGS__>), grid, dim3(router_threads<__VA_ARGS__>()), 0, stream, x, ldx, w, \
                     ldw, bias, n_tokens, hidden, n_expts, logits, ld_logits)
  const bool once = hidden <= 128;  // one or two k-steps: a repeated copy counts
  if (grid.x <= kRtOneRound) {
    if (n_expts <= 32)
      AF3_RT(32, 1, 6);   // 12 KB stages, 6 copies per wave and step
    else if (n_expts <= 64)
      AF3_RT(64, 1, 8);   // 16 KB, 4
    else if (n_expts <= 128)
      AF3_RT(128, 1, 6);  // 24 KB, 3
    else
      AF3_RT(256, 2, 4);  // 40 KB, 5
  } else if (n_expts <= 32) {
    if (once) AF3_RT(32, 1, 2, true);
    else AF3_RT(32, 1, 2);
  } else if (n_expts <= 64) {
    if (once) AF3_RT(64, 1, 2, true);
    else AF3_RT(64, 1, 2);
  } else if (n_expts <= 128) {
    if (once) AF3_RT(128, 1, 2, true);
    else if (hidden < 2048) AF3_RT(128, 1, 2);
    else AF3_RT(128, 1, 3);
  } else if (n_expts <= 192 && hidden >= 512) {
    AF3_RT(192, 3, 2);    // 32 KB, 8
  } else {
    if (once) AF3_RT(256, 2, 2, true);
    else AF3_RT(256, 2, 2);
  }
#undef AF3_RT
  return af3::check_launch("router_logits");
}
