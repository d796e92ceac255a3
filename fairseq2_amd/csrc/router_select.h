// The selection of a token's experts from its logits, the sum of logits that several blocks share, and the bookkeeping of
// dispatch for a few tokens: device functions, because the router's kernels end with them and the expert kernels of a
// decode step begin with them.
#pragma once

#include "common.h"

namespace fs2moe {

__device__ __forceinline__ uint32_t order_key(float v) {
  uint32_t b = __float_as_uint(v);
  if (v != v) return 0xffffffffu;  // NaN ranks above +inf
  if (v == 0.0f) b = 0;            // -0 and +0 tie
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float order_key_inv(uint32_t k) {
  if (k == 0xffffffffu) return __uint_as_float(0x7fc00000u);
  return __uint_as_float((k & 0x80000000u) ? (k ^ 0x80000000u) : ~k);
}

// One wave selects for one token.  v[j] is the logit of expert lane + 64 j (bias included); lane r < K gets the token's
// r-th expert and its weight.
template <int J>
__device__ __forceinline__ void select_experts(const float (&v)[J], int lane, int E, int K, int score_fn, int renorm,
                                               int& expert, float& weight) {
  // Keys of real logits are at least order_key(-inf) = 0x007fffff, so 0 marks "taken / no expert".
  uint32_t key[J];
#pragma unroll
  for (int j = 0; j < J; ++j) key[j] = lane + 64 * j < E ? order_key(v[j]) : 0u;
  int my_e = 0;
  float my_v = 0.f, top_v = 0.f;
  for (int r = 0; r < K; ++r) {
    uint32_t m = key[0];
#pragma unroll
    for (int j = 1; j < J; ++j) m = key[j] > m ? key[j] : m;
    const uint32_t best = wave_max_u32(m);
    // the lowest expert holding `best`: experts lane + 64 j ascend with j first
    int e = 0;
    bool found = false;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const unsigned long long holders = __ballot(key[j] == best);
      if (!found && holders != 0ull) {
        e = 64 * j + (int)__builtin_ctzll(holders);
        found = true;
      }
    }
#pragma unroll
    for (int j = 0; j < J; ++j)
      if (lane + 64 * j == e) key[j] = 0u;
    const float val = order_key_inv(best);
    if (r == 0) top_v = val;
    if (lane == r) {
      my_e = e;
      my_v = val;
    }
  }
  float w;
  if (score_fn == FS2MOE_SCORE_SIGMOID) {
    w = 1.0f / (1.0f + expf(-my_v));
    if (renorm) {
      const float s = wave_sum_f32(lane < K ? w : 0.f);
      w = w / s;
    }
  } else {
    const float ex = expf(my_v - top_v);
    float s;
    if (renorm) {
      s = wave_sum_f32(lane < K ? ex : 0.f);
    } else {
      float part = 0.f;
#pragma unroll
      for (int j = 0; j < J; ++j)
        if (lane + 64 * j < E) part += expf(v[j] - top_v);
      s = wave_sum_f32(part);
    }
    w = ex / s;
  }
  expert = my_e;
  weight = w;
}

// The same, written to memory.
template <int J>
__device__ __forceinline__ void select_topk(const float (&v)[J], int lane, int t, int E, int K,
                                            int score_fn, int renorm,
                                            int32_t* __restrict__ topk_idx,
                                            float* __restrict__ topk_w, int* chosen = nullptr, float* weight = nullptr) {
  int my_e;
  float w;
  select_experts<J>(v, lane, E, K, score_fn, renorm, my_e, w);
  if (lane < K) {
    topk_idx[(size_t)t * K + lane] = my_e;
    topk_w[(size_t)t * K + lane] = w;
  }
  if (chosen != nullptr) *chosen = my_e;
  if (weight != nullptr) *weight = w;
}

// Blocks sharing a token tile, at most: every bf16 D up to 5120 takes one step a block (2560 with more than 128
// experts), longer rows two.  The finishing kernel issues this many loads a lane whatever D, those past the
// last block masked off.  With 32 of them D 6144 to 8192 would take one step as well (64 tokens, 16 to 128
// experts 9.7-13.7 -> 7.9-13.4 us, with the norm 17.6-25.2 -> 12.3-19.3), but a layer's step of any smaller D
// took longer: D 2048, 128 experts 32.7 -> 33.7 us at one token, D 576, 16 experts 60.5 -> 62.0 at 4000.
constexpr int kMaxSlices = 20;

// Second half of the split router: one wave per token adds the `slices` partial logits in
// ascending order, then the bias, and selects.
template <int J>
__device__ __forceinline__ void finish_logits(const float* __restrict__ partial, int slices,
                                              const float* __restrict__ bias, int t, int T, int E, float (&v)[J]) {
  const int lane = lane_id();
  // all loads first (at most kMaxSlices of them per expert), then the sums in ascending order
  float p[kMaxSlices][J], b[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int e = lane + 64 * j;
    b[j] = (bias != nullptr && e < E) ? bias[e] : 0.f;
#pragma unroll
    for (int s = 0; s < kMaxSlices; ++s)
      p[s][j] = (s < slices && e < E) ? partial[((size_t)s * T + t) * E + e] : 0.f;
  }
#pragma unroll
  for (int j = 0; j < J; ++j) {
    float sum = p[0][j];
#pragma unroll
    for (int s = 1; s < kMaxSlices; ++s) sum += p[s][j];
    v[j] = sum + b[j];
  }
}
template <int J>
__device__ __forceinline__ void finish_token(const float* __restrict__ partial, int slices,
                                             const float* __restrict__ bias, int t, int T, int E, int K,
                                             int score_fn, int renorm, int32_t* topk_idx, float* topk_w,
                                             float* logits, int* chosen, float* weight) {
  const int lane = lane_id();
  float v[J];
  finish_logits<J>(partial, slices, bias, t, T, E, v);
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (logits != nullptr && lane + 64 * j < E) logits[(size_t)t * E + lane + 64 * j] = v[j];
  select_topk<J>(v, lane, t, E, K, score_fn, renorm, topk_idx, topk_w, chosen, weight);
}

// Dispatch of at most 32 tokens whose selection is in registers and LDS, by all THREADS threads of a block: wave w holds
// tokens w + THREADS / 64 i, lane k < K of it the token's k-th expert and weight, and s_bits a word per expert with a bit
// per token (complete: a barrier has been passed).  s_off [64 J + 1] and s_wave_tot [J] are scratch.
template <int J, int THREADS, int TPW>
__device__ __forceinline__ void dispatch_finished(const uint32_t* s_bits, int32_t* s_off, int32_t* s_wave_tot,
                                                  const int (&chosen)[TPW], const float (&weight)[TPW], int T, int E, int K,
                                                  int tile_m, int64_t max_rows, int32_t* __restrict__ counts,
                                                  int32_t* __restrict__ offsets, int32_t* __restrict__ perm,
                                                  int32_t* __restrict__ inv_perm, float* __restrict__ row_w) {
  constexpr int NW = THREADS / kWave;
  const int tid = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  // counts and tile-padded offsets: a thread per expert, a scan over the J waves that hold them
  int cnt = 0, padded = 0, incl = 0;
  if (wave < J) {
    cnt = __popc(s_bits[tid]);
    padded = (cnt + tile_m - 1) / tile_m * tile_m;
    incl = padded;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(incl, off, kWave);
      if (lane >= off) incl += v;
    }
    if (lane == 63) s_wave_tot[wave] = incl;
  }
  __syncthreads();
  if (wave < J) {
    int base = 0;
    for (int w = 0; w < wave; ++w) base += s_wave_tot[w];
    s_off[tid] = base + incl - padded;
    if (tid == 64 * J - 1) s_off[64 * J] = base + incl;
    if (tid < E) {
      counts[tid] = cnt;
      offsets[tid] = base + incl - padded;
      if (tid == E - 1) offsets[E] = base + incl;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int tl = wave + NW * i;
    if (tl >= T || lane >= K) continue;
    const int row = s_off[chosen[i]] + __popc(s_bits[chosen[i]] & ((1u << tl) - 1u));
    inv_perm[(size_t)tl * K + lane] = row;
    perm[row] = tl;
    // (for kernels that scale a row by its routing weight while they read it through perm)
    if (row_w != nullptr) row_w[row] = weight[i];
  }
  // padding rows, then the rows beyond the last expert's
  if (tid < E)
    for (int r = s_off[tid] + cnt; r < s_off[tid + 1]; ++r) perm[r] = -1;
  for (int64_t r = (int64_t)s_off[64 * J] + tid; r < max_rows; r += THREADS) perm[r] = -1;
}

}  // namespace fs2moe
