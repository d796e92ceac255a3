// Grouped SwiGLU products for a handful of rows per expert, bf16 weights in the reference layout.
//
// A decode step of one to eight sequences gives every active expert at most that many rows: the
// layer is then a stream over the active experts' weights, each weight used once per row.  The
// throughput kernel handles such an expert as a tile of 256 channels walked through all of K by one
// block, i.e. a chain of K / 64 round trips on one CU with the matrix pipe all but idle (8 experts x
// 6 tiles keep 48 of 256 CUs busy for 32 us).  Here the weights never pass through LDS or the matrix
// pipe: a lane loads 16 bytes (8 channels of one k row, as they lie in memory, (K, N) with N
// contiguous), multiplies them with that k's activation of each row on the vector ALUs and keeps
// R x 8 sums (twice that for the fused gate/up product).  A block owns 64 channels of one expert:
// its eight waves split K, a wave's eight lane groups split it again (a load instruction covers
// 8 lane groups x 4 k rows of 128 contiguous bytes), and the partial sums are added in a fixed
// order: lane groups by exchange within the wave, waves through LDS.  The expert's rows sit in LDS
// as they lie in memory; a lane reads the 4 k it needs of each row with one 8-byte read.
//
// R (1, 2 or 4) is the most rows of one expert taken per pass: a template parameter that bounds the
// registers (rows an expert does not have are skipped); an expert with more rows than R is walked
// again for every further R rows (correct for any count, meant for counts up to R).  From 5 rows per
// expert on the arithmetic no longer hides behind the stream and the GEMM tiles are faster.
#pragma once

#include <type_traits>

#include "common.h"
#include "router_select.h"

namespace fs2moe {
namespace gemv {
constexpr int COLS = 64;          // channels per block
// waves per block: a block is a short chain of round trips to memory, so K is split over eight
// waves (with four, one token took 47 instead of 44 us and four tokens 71 instead of 61)
constexpr int waves(int R) { return 8; }
constexpr int threads(int R) { return 64 * waves(R); }
constexpr int MAX_LDS_BYTES = 144 * 1024;  // (160 KB less the kernel's own partial sums, 16 KB at most)
constexpr int MAX_LDS_SELECT = MAX_LDS_BYTES - 6 * 1024;  // (less what a kernel that selects keeps of it)
inline bool fits(int K, int R) { return (int64_t)K * R * 2 <= MAX_LDS_BYTES; }
// Steps of K (256 rows a block) whose loads a wave has in flight: 4 with one or two rows, 2 with four
// (registers).  DEEP: 8, for the single product with one or two rows over a
// long K, where a block is a chain of K / 256 / U round trips (Mixtral's down projection, K 14336:
// the layer at one token 225 -> 178 us, at two 286 -> 251; a short K would only issue loads that it
// then masks: Qwen3's K of 768 is three steps, and two tokens took 54 instead of 48 us with 8).
// The sums do not depend on it: a lane adds its products in the same order.
constexpr int steps_in_flight(bool dual, int R, bool deep) { return R > 2 ? 2 : (deep && !dual) ? 8 : 4; }
inline bool deep_applies(int K, int R) { return R <= 2 && K >= 4096; }
// (one expert's matrix is addressed with 32-bit byte offsets, by up to 4096 rows past its end)
inline bool offsets_fit(int D, int F) {
  const int64_t lo = D < F ? D : F, hi = D < F ? F : D;
  return (lo + 4096) * hi * 2 < 0xffffffffll && (hi + 4096) * lo * 2 < 0xffffffffll;
}
}  // namespace gemv
// One expert's matrix as a buffer: a row past its end reads as zeros, without memory traffic.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t expert_matrix(const uint16_t* B, int e, int K, int N) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(B + (size_t)e * K * N), 0,
                                           (int)((uint32_t)K * (uint32_t)N * 2u), 0x00020000);
}

// The n-th expert that has rows, -1 when there are fewer (wave-uniform; every wave works it out for
// itself from the counts, without LDS or a barrier: E <= 256 is four ballots).  A block takes the
// blockIdx.y-th such expert instead of expert blockIdx.y: blocks of experts without rows would end at
// once wherever they are, but numbered this way the blocks that work are contiguous in launch order
// whatever the experts' numbers, and consecutive blocks go to consecutive XCDs.  With the real routing
// of 12 tokens (24 experts active, scattered over 128) the blocks of the block-per-CU kernel below
// crowded on some XCDs and its pair of launches took 73 instead of 54 us.  The grid holds about as many
// blocks as run at once, and a block goes on to the expert gridDim.y further: with a block for every
// expert there may be, the last of those without rows began a microsecond or two after the others' end.
__device__ __forceinline__ int nth_active_expert(const int32_t* __restrict__ counts, int E, int n) {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));  // (nothing of this is kept from one expert to the next)
  int c[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = lane + 64 * j;
    c[j] = counts[i < E ? i : 0];
  }
  int e = -1, seen = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const unsigned long long act = __ballot(lane + 64 * j < E && c[j] > 0);
    const int before = __popcll(act & ((1ull << lane) - 1ull));
    const unsigned long long hit = __ballot(((act >> lane) & 1ull) != 0ull && seen + before == n);
    if (e < 0 && hit != 0ull) e = 64 * j + (int)__builtin_ctzll(hit);
    seen += __popcll(act);
  }
  return e;
}

// ---------------------------------------------------------------------------------------------------
// The shared expert (a dense SwiGLU, weights as nn.Linear holds them: (N, K) with K contiguous) for
// up to 16 rows: at a decode step its three matrices are streamed once like an expert's, and the
// GEMM tiles make that a chain of K / 64 round trips per tile (Llama-4 Scout, one token: 172 us for
// 252 MB).  Here 16 bytes of a weight row ARE eight k of one channel, which is what
// v_mfma_f32_16x16x32_bf16 takes from lane (n = l % 16, g = l / 16) as it stands; the matching lane
// (m = l % 16, g) loads the same eight k of row m straight from memory (the rows stay in L2; a row
// the call does not have repeats the last one, its results are not stored).  A block owns 16
// channels, its eight waves split K in steps of 32 and add their sums in LDS in ascending order.
namespace dgemv {
constexpr int WAVES = 8, THREADS = WAVES * 64;
constexpr int U = 8;  // steps of 32 k a wave has in flight
constexpr int MAX_ROWS = 16;
constexpr int red_bytes(bool dual) { return WAVES * (dual ? 2 : 1) * 64 * 16; }
}  // namespace dgemv

// DUAL: C[r, n] = SiLU(A[r] . B0[n]) * (A[r] . B1[n]); else C[r, n] = A[r] . B0[n].
// A [T][lda], B0/B1 [N][K], C [T][ldc]; T <= 16; K and N multiples of 8.  grid: ceil(N / 16).
// red: LDS of red_bytes(DUAL).
template <bool DUAL, bool NT>
__device__ __forceinline__ void dense_gemv_block(
    const uint16_t* __restrict__ A, int lda, const uint16_t* __restrict__ B0,
    const uint16_t* __restrict__ B1, uint16_t* __restrict__ C, int ldc, int K, int N, int T, int block, uint8_t* lds) {
  using namespace dgemv;
  constexpr int M = DUAL ? 2 : 1;
  f32x4(*red)[M][64] = reinterpret_cast<f32x4(*)[M][64]>(lds);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int n0 = block * 16;
  const int n = n0 + r16 < N ? n0 + r16 : N - 1;  // a channel past N repeats the last one: not stored
  const int row = r16 < T ? r16 : T - 1;
  const uint16_t* w0 = B0 + (size_t)n * K;
  const uint16_t* w1 = DUAL ? B1 + (size_t)n * K : w0;
  const uint16_t* xr = A + (size_t)row * lda;
  f32x4 acc[M];
#pragma unroll
  for (int m = 0; m < M; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  // step s of the block is the 32 k from 32 s; wave w takes the steps w, w + 8, ..
  for (int s0 = wave; s0 * 32 < K; s0 += WAVES * U) {
    u32x4 wq[U][M], xq[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = (s0 + u * WAVES) * 32 + g * 8;
      const int kk = k < K ? k : 0;  // K is a multiple of 8: the lane's eight k are in or out together
      wq[u][0] = load_weights<NT>(w0 + kk);
      if (DUAL) wq[u][M - 1] = load_weights<NT>(w1 + kk);
      xq[u] = *reinterpret_cast<const u32x4*>(xr + kk);
    }
    // (all the loads are issued before the first is waited for)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = (s0 + u * WAVES) * 32 + g * 8;
      u32x4 xv = xq[u];
      if (k >= K) xv = u32x4{0u, 0u, 0u, 0u};
      const bf16x8 xop = __builtin_bit_cast(bf16x8, xv);
#pragma unroll
      for (int m = 0; m < M; ++m)
        acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wq[u][m]), xop,
                                                         acc[m], 0, 0, 0);
    }
  }
#pragma unroll
  for (int m = 0; m < M; ++m) red[wave][m][lane] = acc[m];
  __syncthreads();
  if (wave != 0) return;
  // lane (row m = l % 16, q = l / 16) holds channels n0 + 4 q + i, i = 0..3
  f32x4 sum[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    sum[m] = red[0][m][lane];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sum[m] += red[w][m][lane];
  }
  const int nc = n0 + 4 * g;
  if (r16 < T && nc < N) {  // N is a multiple of 8: four channels are in or out together
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = DUAL ? silu_f32(sum[0][i]) * sum[M - 1][i] : sum[0][i];
    u32x2 o = {(uint32_t)f32_to_bf16_bits(v[0]) | ((uint32_t)f32_to_bf16_bits(v[1]) << 16),
               (uint32_t)f32_to_bf16_bits(v[2]) | ((uint32_t)f32_to_bf16_bits(v[3]) << 16)};
    *reinterpret_cast<u32x2*>(C + (size_t)r16 * ldc + nc) = o;
  }
}
template <bool DUAL, bool NT>
__global__ __launch_bounds__(dgemv::THREADS) void dense_gemv_bf16_kernel(
    const uint16_t* __restrict__ A, int lda, const uint16_t* __restrict__ B0,
    const uint16_t* __restrict__ B1, uint16_t* __restrict__ C, int ldc, int K, int N, int T) {
  __shared__ __attribute__((aligned(16))) uint8_t red[dgemv::red_bytes(DUAL)];
  dense_gemv_block<DUAL, NT>(A, lda, B0, B1, C, ldc, K, N, T, (int)blockIdx.x, red);
}
// The same product of the shared expert in the launch of the routed ones: `blocks` blocks of it (0: none).
struct DenseBeside {
  const uint16_t *A, *B0, *B1;
  uint16_t* C;
  int K, N, T, blocks;
};
template <bool DUAL>
__device__ __forceinline__ void dense_beside_block(const DenseBeside& d, int block, uint8_t* lds) {
  dense_gemv_block<DUAL, false>(d.A, d.K, d.B0, d.B1, d.C, d.N, d.K, d.N, d.T, block, lds);
}

// SELECT 2 or 4 (gate/up): the kernel begins with what router_finish_tile_kernel does, for at most 16 tokens and 64 SELECT
// experts.  Every block adds the partial logits, selects and keeps a word per expert with a bit per token in LDS, from which
// its experts, their rows and those rows' tokens follow without a look at memory; the last block of the grid, which has the
// least to stream, writes what the kernels behind it read.  A launch of one block is a boundary and a chain of round trips
// while the chip waits (6 to 7 us); here it is 2 us in front of the stream, as its three look-ups (counts, offsets, tokens)
// are gone.  Each block pays them, so there is one a CU, which takes (expert, channel block) pairs in turn: with a block for
// every pair 4 tokens took 70 us.  us of the layer under a graph, D 2048, F 768, top-8 of 128, with the launch and without:
//   1 token 43.7, 40.6    2 53.4, 49.7    4 63.5, 59.6    8 75.3, 72.2    12 78.3, 76.5    16 81.6, 79.7
// 3 of D 1024, F 1408, top-4 of 60, rows scaled 47.5, 44.0; 1 of D 4096, F 14336, top-2 of 8 173.3, 169.8.
struct Selected {
  uint32_t bits[256];
  float weight[16][FS2MOE_MAX_TOP_K];  // by token and slot, and their experts
  int16_t expert[16][FS2MOE_MAX_TOP_K];
  int32_t off[257], wave_tot[4];
};
template <int SELECT, int THREADS>
__device__ __forceinline__ void select_for_block(Selected& s, const Selection& sel, int E, bool writes) {
  constexpr int NW = THREADS / kWave, TPW = 16 / NW;
  const int tid = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  static_assert(64 * SELECT <= THREADS && SELECT <= 4, "a thread per expert");
  if (tid < 64 * SELECT) s.bits[tid] = 0u;
  __syncthreads();
  int chosen[TPW];
  float weight[TPW];
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int t = wave + NW * i;
    chosen[i] = 0;
    weight[i] = 0.f;
    if (t >= sel.T) continue;  // wave-uniform
    float v[SELECT];
    finish_logits<SELECT>(sel.partial, sel.slices, sel.bias, t, sel.T, E, v);
    select_experts<SELECT>(v, lane, E, sel.K, sel.score_fn, sel.renormalize, chosen[i], weight[i]);
    if (lane < sel.K) {
      atomicOr(&s.bits[chosen[i]], 1u << t);
      s.weight[t][lane] = weight[i];
      s.expert[t][lane] = (int16_t)chosen[i];
      if (writes) {
        sel.topk_idx[(size_t)t * sel.K + lane] = chosen[i];
        sel.topk_w[(size_t)t * sel.K + lane] = weight[i];
      }
    }
  }
  __syncthreads();
  if (writes)
    dispatch_finished<SELECT, THREADS, TPW>(s.bits, s.off, s.wave_tot, chosen, weight, sel.T, E, sel.K, sel.tile_m,
                                            sel.max_rows, sel.counts, sel.offsets, sel.perm, sel.inv_perm, sel.row_w);
}
// The n-th expert with rows (-1: there is none) with its number of rows and its first row.
template <int SELECT>
__device__ __forceinline__ int nth_selected_expert(const Selected& s, int tile_m, int n, int& cnt, int& off) {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));  // (as in nth_active_expert)
  int e = -1, seen = 0, c[SELECT];
#pragma unroll
  for (int j = 0; j < SELECT; ++j) {
    c[j] = __popc(s.bits[lane + 64 * j]);
    const unsigned long long act = __ballot(c[j] > 0);
    const int before = __popcll(act & ((1ull << lane) - 1ull));
    const unsigned long long hit = __ballot(((act >> lane) & 1ull) != 0ull && seen + before == n);
    if (e < 0 && hit != 0ull) e = 64 * j + (int)__builtin_ctzll(hit);
    seen += __popcll(act);
  }
  if (e < 0) return e;
  int rows = 0;
#pragma unroll
  for (int j = 0; j < SELECT; ++j) rows += lane + 64 * j < e ? (c[j] + tile_m - 1) / tile_m * tile_m : 0;
  off = wave_sum_i32(rows);
  cnt = __builtin_amdgcn_readfirstlane(__popc(s.bits[e]));
  return e;
}
static_assert(sizeof(Selected) <= 6 * 1024, "left out of MAX_LDS_SELECT");
// The shared expert's product in the routed ones' launch: its own two launches had each a boundary and a round trip or two
// while most of the chip waited, and the routed ones' blocks do not fill it either.  us of the layer under a graph with the
// launches and without: 1 and 8 tokens of D 2048, F 768, top-8 of 128 53.8, 41.2 and 85.5, 70.6; 2 and 12 of D 1024, F 1408,
// top-4 of 60 53.3, 42.8 and 101.9, 85.8; 6 of D 4096, F 4096, top-2 of 16 242, 233.  (One whose weights are loaded past the
// caches has launches of its own, as has one of 192 MB and more, which runs beside the whole routed path.)
// What a block has to do of it, in front of its own.  SELECT (blocks that stay): blocks d, d + grid,
// .. of it, and the routed experts' pairs go on where those end; returns the block's first pair.  Else the first rows of the
// grid are theirs; returns how many, or -1 in such a block.
template <bool DUAL, bool SELECT>
__device__ __forceinline__ int dense_of_grid(const DenseBeside& dense, uint8_t* lds) {
  const int grid = (int)gridDim.x;
  if constexpr (SELECT) {
    int b = (int)blockIdx.x;
    for (; b < dense.blocks; b += grid) {
      if (b >= grid) __syncthreads();  // (the sums of the block before)
      dense_beside_block<DUAL>(dense, b, lds);
    }
    return b - dense.blocks;
  } else if constexpr (DUAL) {
    return 0;  // (gate/up goes with the selection only)
  } else {
    const int rows = (dense.blocks + grid - 1) / grid;
    if ((int)blockIdx.y >= rows) return rows;
    const int b = (int)blockIdx.y * grid + (int)blockIdx.x;
    if (b < dense.blocks) dense_beside_block<DUAL>(dense, b, lds);
    return -1;
  }
}
// The token of the expert's r-th row, and the weight of that pair.
__device__ __forceinline__ int selected_token(uint32_t bits, int r) {
  for (int i = 0; i < r; ++i) bits &= bits - 1u;
  return (int)__builtin_ctz(bits);
}
__device__ __forceinline__ float selected_weight(const Selected& s, int t, int e, int K) {
  const int lane = lane_id(), k = lane < K ? lane : 0;
  const unsigned long long hit = __ballot(s.expert[t][k] == e);
  return s.weight[t][(int)__builtin_ctzll(hit)];
}

// DUAL: C[r, n] = SiLU(A[r] . B0[:, n]) * (A[r] . B1[:, n]); else C[r, n] = A[r] . B0[:, n].
// A rows are read through row_map when it is given (row r of the expert is A[row_map[offset + r]]),
// and multiplied by row_w[offset + r] on the way into LDS when that is given (rounded to bf16: the
// bits dispatch's scaled row copy would have held).
// grid: (ceil(N / 64), as many experts at a time as fill the chip).  K a multiple of 4, N a multiple of 8.
// NT: the weights are loaded past the caches (load_once).
template <bool DUAL, int R, bool NT, bool DEEP = false, int SELECT = 0>
__global__ __launch_bounds__(gemv::threads(R)) void glu_gemv_bf16_kernel(
    const uint16_t* __restrict__ A, const int32_t* __restrict__ row_map,
    const float* __restrict__ row_w, int lda,
    const uint16_t* __restrict__ B0, const uint16_t* __restrict__ B1, uint16_t* __restrict__ C,
    int ldc, int K, int N, const int32_t* __restrict__ counts,
    const int32_t* __restrict__ offsets, int E, const Selection sel, const DenseBeside dense) {
  using namespace gemv;
  constexpr int M = DUAL ? 2 : 1;
  constexpr int NW = waves(R), THREADS = threads(R);
  constexpr int KSTEP = NW * 32;  // k rows per block and step: NW waves x 8 lane groups x 4
  extern __shared__ __attribute__((aligned(16))) uint8_t gemv_smem[];
  uint16_t* xs = reinterpret_cast<uint16_t*>(gemv_smem);  // [R][K]
  __shared__ float red[NW][M][R][COLS];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ks = lane >> 3, cc = lane & 7;
  const int dense_rows = dense_of_grid<DUAL, SELECT != 0>(dense, gemv_smem);
  if (dense_rows < 0) return;
  __shared__ std::conditional_t<SELECT != 0, Selected, char> chosen;
  if constexpr (SELECT != 0)
    select_for_block<SELECT, THREADS>(chosen, sel, E, blockIdx.x == gridDim.x - 1);
  const int col_blocks = (N + COLS - 1) / COLS;
  const int items_at_once = SELECT != 0 ? (int)gridDim.x : (int)gridDim.y - dense_rows;
  for (int item = SELECT != 0 ? dense_rows : (int)blockIdx.y - dense_rows;; item += items_at_once) {
  int e, cnt, off, col_block;
  if constexpr (SELECT != 0) {
    const int nth = item / col_blocks;
    col_block = item - nth * col_blocks;
    e = nth_selected_expert<SELECT>(chosen, sel.tile_m, nth, cnt, off);
    if (e < 0) return;
  } else {
    col_block = (int)blockIdx.x;
    e = nth_active_expert(counts, E, item);
    if (e < 0) return;
    cnt = counts[e];
    off = offsets[e];
  }
  const __amdgpu_buffer_rsrc_t w_rsrc[2] = {expert_matrix(B0, e, K, N), expert_matrix(DUAL ? B1 : B0, e, K, N)};
  const int col = col_block * COLS + cc * 8;
  const bool col_ok = col < N;  // N is a multiple of 8: the lane's eight channels are in or out together
  // U steps of K are in flight, each loaded into the registers of the one U before it as soon as that has
  // been multiplied.  The first of them are issued before the rows are even looked up: they need only the
  // expert's number, and a decode step's block is a chain of round trips (one token, D 2048 / F 768: the
  // pair 23.1 -> 20.4 us).
  constexpr int U = gemv::steps_in_flight(DUAL, R, DEEP);
  u32x4 wv[U][M][4];
  // (a lane's four rows of a step are in or out of the matrix together, so that the first one's offset
  // decides; the others add a scalar to it)
  uint32_t at;  // the lane's place in the next step
  auto rewind = [&]() {
    uint32_t row = (uint32_t)(wave * 32 + ks * 4);
    asm volatile("" : "+v"(row));  // (else addresses are computed in front of the passes and kept)
    at = (row * (uint32_t)N + (uint32_t)(col_ok ? col : 0)) * 2u;
  };
  auto load_step = [&](int set) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int m = 0; m < M; ++m)
        wv[set][m][j] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc[m], at, j * N * 2, NT ? kNonTemporal : 0);
    at += (uint32_t)KSTEP * (uint32_t)N * 2u;
  };
  const int steps = (K + KSTEP - 1) / KSTEP;

  for (int r0 = 0; r0 < cnt; r0 += R) {
    // (where rows are looked up, half of the steps go in front of that and half behind the rows' loads;
    // the down projection's rows lie in order and come from L2: they go first)
    constexpr int FRONT = DUAL ? U / 2 : 0;
    rewind();
#pragma unroll
    for (int u = 0; u < FRONT; ++u) load_step(u);
    __builtin_amdgcn_sched_barrier(0);
    // ---- the pass's rows -> LDS (rows past the expert's count as zeros) ---------------------------
    __syncthreads();  // the previous pass's reads of xs and red are over
    const int kchunks = K / 4;    // 8-byte pieces per row
    // (rows the expert does not have are skipped, block-uniformly: R only bounds the registers; where
    // a row lies is wave-uniform, and looked up by scalar loads, which do not wait for the vector ones)
    const int rcnt = __builtin_amdgcn_readfirstlane(cnt - r0 < R ? cnt - r0 : R);
    size_t src[R];
    float rw[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if constexpr (SELECT != 0) {
        const int t = selected_token(__builtin_amdgcn_readfirstlane(chosen.bits[e]), r0 + (r < rcnt ? r : 0));
        src[r] = (size_t)t * lda;
        rw[r] = row_w != nullptr ? selected_weight(chosen, t, e, sel.K) : 1.f;
        continue;
      }
      const int row = off + r0 + (r < rcnt ? r : 0);
      src[r] = (size_t)(row_map != nullptr ? row_map[row] : row) * lda;
      rw[r] = row_w != nullptr ? row_w[row] : 1.f;
    }
    constexpr int AHEAD = R > 2 ? 1 : 2;  // pieces of each row in flight per thread
    u32x2 v[R][AHEAD];
    auto load_rows = [&](int c0) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
          const int c = c0 + i * THREADS;
          v[r][i] = *reinterpret_cast<const u32x2*>(A + src[r] + 4 * (c < kchunks ? c : 0));
        }
    };
    auto store_rows = [&](int c0) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
          const int c = c0 + i * THREADS;
          u32x2 q = v[r][i];
          if (r >= rcnt) q = u32x2{0u, 0u};
          if (row_w != nullptr) q = u32x2{scale_bf16x2(q[0], rw[r]), scale_bf16x2(q[1], rw[r])};
          if (c < kchunks) *reinterpret_cast<u32x2*>(xs + (size_t)r * K + 4 * c) = q;
        }
    };
    load_rows(tid);
    // (behind the first of the rows, which are waited for first)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = FRONT; u < U; ++u) load_step(u);
    __builtin_amdgcn_sched_barrier(0);
    store_rows(tid);
    for (int c0 = tid + AHEAD * THREADS; c0 < kchunks; c0 += AHEAD * THREADS) {
      load_rows(c0);
      store_rows(c0);
    }
    lds_barrier();

    // ---- the stream over K --------------------------------------------------------------------------
    float acc[M][R][8];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[m][r][c] = 0.f;
    // (the last U steps load nothing: loads past K's end cost as much of the CU's load path as others)
    auto multiply = [&](int s0, auto more) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k0 = (s0 + u) * KSTEP + wave * 32 + ks * 4;
        const bool k_ok = k0 < K;  // K is a multiple of 4: the lane's four rows are in or out together
        const int kk = k_ok ? k0 : 0;
        float xv[R][4];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          if (r < rcnt) {
            const u32x2 q = *reinterpret_cast<const u32x2*>(xs + (size_t)r * K + kk);
            xv[r][0] = k_ok ? __uint_as_float(q[0] << 16) : 0.f;
            xv[r][1] = k_ok ? __uint_as_float(q[0] & 0xffff0000u) : 0.f;
            xv[r][2] = k_ok ? __uint_as_float(q[1] << 16) : 0.f;
            xv[r][3] = k_ok ? __uint_as_float(q[1] & 0xffff0000u) : 0.f;
          }
        }
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            float wf[8];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              wf[2 * c] = __uint_as_float(wv[u][m][j][c] << 16);
              wf[2 * c + 1] = __uint_as_float(wv[u][m][j][c] & 0xffff0000u);
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
              if (r < rcnt) {
#pragma unroll
                for (int c = 0; c < 8; ++c) acc[m][r][c] += xv[r][j] * wf[c];
              }
            }
          }
        // (without the fences the compiler moves every load down to its first use and waits for each
        // one there: one round trip per load)
        if constexpr (decltype(more)::value) {
          __builtin_amdgcn_sched_barrier(0);
          load_step(u);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    int s0 = 0;
    for (; s0 + U < steps; s0 += U) multiply(s0, std::true_type{});
    multiply(s0, std::false_type{});

    // ---- lane groups (fixed order: exchange distances 8, 16, 32), then waves through LDS ------------
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (r < rcnt) {
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            float v = acc[m][r][c];
            v += __shfl_xor(v, 8, kWave);
            v += __shfl_xor(v, 16, kWave);
            v += __shfl_xor(v, 32, kWave);
            acc[m][r][c] = v;
          }
        }
      }
    if (ks == 0) {
#pragma unroll
      for (int m = 0; m < M; ++m)
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int c = 0; c < 8; ++c) red[wave][m][r][cc * 8 + c] = acc[m][r][c];
    }
    __syncthreads();
    for (int i = tid; i < R * COLS; i += THREADS) {
      const int r = i / COLS, c = i - r * COLS;
      const int n = col_block * COLS + c;
      if (r0 + r >= cnt || n >= N) continue;
      float g = 0.f, u = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        g += red[w][0][r][c];
        if (DUAL) u += red[w][M - 1][r][c];
      }
      if (DUAL) g = silu_f32(g) * u;
      C[(size_t)(off + r0 + r) * ldc + n] = f32_to_bf16_bits(g);
    }
  }
  }
}


// ---------------------------------------------------------------------------------------------------
// The same stream for 5 to 16 rows per expert, with the arithmetic on the matrix pipe and still no
// LDS transposition of the weights.  v_mfma_f32_16x16x32_bf16 wants, per lane, eight k of ONE
// channel; a lane's 16-byte load holds eight channels of ONE k.  But the 32 k slots of the
// instruction are just 32 products summed per (channel, row) pair: which k sits in which slot is
// free as long as both operands agree.  So a lane (c16 = l % 16, g = l / 16) loads its eight
// channels 8 c16 .. 8 c16 + 7 at eight k rows (two steps of four consecutive rows), and one byte
// permute per pair of rows turns that 8 x 8 block of its OWN registers into eight operands, one per
// channel, each holding the lane's eight k in its eight slots.  MFMA number c of a step then multiplies
// channels {8 r + c : r = 0..15} (one per lane of a group) with up to 16 rows of the expert over
// 4 groups x 8 k, and the lane (row m = l % 16, q = l / 16) ends up with channels 8 (4 q + i) + c,
// i = 0..3.  The rows' operand is what lies in LDS: the 2 x 4 consecutive k of row m.
//
// A block owns 128 channels of one expert; its eight waves split K (a step of the block is 128 k
// rows) and their partial sums meet in LDS in a fixed order ((0+4)+(2+6))+((1+5)+(3+7)).  XR (8 or
// 16) is how many rows are staged in LDS: a pass takes up to XR rows, an expert with more is walked
// again.  Rows lie K + 4 elements apart so that the sixteen rows' reads fall into different banks.
namespace gemv16 {
constexpr int COLS = 128;     // channels per block: 16 lanes x 8
constexpr int WAVES = 8, THREADS = WAVES * 64;
constexpr int KSTEP = WAVES * 16;  // k rows per step of the block: waves x 4 lane groups x 4
constexpr int MAX_LDS_BYTES = 160 * 1024, MAX_LDS_SELECT = MAX_LDS_BYTES - 6 * 1024;
__host__ __device__ inline int stride(int K) { return K + 4; }
inline size_t lds_bytes(int K, int XR, bool dual) {
  const size_t xs = ((size_t)XR * stride(K) + 4) * 2;
  const size_t red = (size_t)4 * (dual ? 2 : 1) * 32 * 64 * 4;
  return xs > red ? xs : red;
}
inline bool fits(int K, int XR) { return lds_bytes(K, XR, true) <= (size_t)MAX_LDS_BYTES; }
}  // namespace gemv16

// Arguments as glu_gemv_bf16_kernel.  grid: (ceil(N / 128), experts at a time).  K and N multiples of 8.
// (The second launch bound is waves per SIMD: the single product is held to 128 registers so that
// two blocks share a CU -- the down projection of 20 active experts is 320 blocks, which at one block
// per CU ran as a full round and a quarter-full one: 4 us of 75 at 8 tokens.)
template <bool DUAL, int XR, bool NT, int SELECT = 0>
__global__ __launch_bounds__(gemv16::THREADS, DUAL ? 2 : 4) void glu_gemv16_bf16_kernel(
    const uint16_t* __restrict__ A, const int32_t* __restrict__ row_map,
    const float* __restrict__ row_w, int lda,
    const uint16_t* __restrict__ B0, const uint16_t* __restrict__ B1, uint16_t* __restrict__ C,
    int ldc, int K, int N, const int32_t* __restrict__ counts,
    const int32_t* __restrict__ offsets, int E, const Selection sel, const DenseBeside dense) {
  using namespace gemv16;
  constexpr int M = DUAL ? 2 : 1;
  constexpr int SETS = 2;  // pairs of steps in flight: 32 (DUAL) or 16 loads per lane
  extern __shared__ __attribute__((aligned(16))) uint8_t gemv16_smem[];
  uint16_t* xs = reinterpret_cast<uint16_t*>(gemv16_smem);  // [XR][K + 4], then 4 zeros
  float* red = reinterpret_cast<float*>(gemv16_smem);       // [4][M][32][64], after the stream

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ldx = stride(K);
  const int dense_rows = dense_of_grid<DUAL, SELECT != 0>(dense, gemv16_smem);
  if (dense_rows < 0) return;
  __shared__ std::conditional_t<SELECT != 0, Selected, char> chosen;
  if constexpr (SELECT != 0)
    select_for_block<SELECT, THREADS>(chosen, sel, E, blockIdx.x == gridDim.x - 1);
  const int col_blocks = (N + COLS - 1) / COLS;
  const int items_at_once = SELECT != 0 ? (int)gridDim.x : (int)gridDim.y - dense_rows;
  for (int item = SELECT != 0 ? dense_rows : (int)blockIdx.y - dense_rows;; item += items_at_once) {
  int e, cnt, off, col_block;
  if constexpr (SELECT != 0) {
    const int nth = item / col_blocks;
    col_block = item - nth * col_blocks;
    e = nth_selected_expert<SELECT>(chosen, sel.tile_m, nth, cnt, off);
    if (e < 0) return;
  } else {
    col_block = (int)blockIdx.x;
    e = nth_active_expert(counts, E, item);
    if (e < 0) return;
    cnt = counts[e];
    off = offsets[e];
  }
  // the expert's matrices as buffers, a lane's place in them as a 32-bit byte offset (one register per
  // address, shared by gate and up)
  const __amdgpu_buffer_rsrc_t w_rsrc[2] = {expert_matrix(B0, e, K, N), expert_matrix(DUAL ? B1 : B0, e, K, N)};
  const int pairs = (K + 2 * KSTEP - 1) / (2 * KSTEP);

  for (int r0 = 0; r0 < cnt; r0 += XR) {
    // (everything a lane derives from its number, anew for each pass: kept across the passes it costs
    // the registers that the loads need, and a value spilled to memory is read back behind those loads)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, c16 = lane & 15, g = lane >> 4;
    const int col = col_block * COLS + c16 * 8;
    // (N is a multiple of 8: the lane's eight channels are in or out together)
    const uint32_t lane_col = (uint32_t)(col < N ? col : 0);
    const bool row_ok = c16 < XR;  // row m = c16 of the pass, if it is staged; else, and past K, zeros
    const int xzero = XR * ldx, xrow = c16 * ldx, xend = row_ok ? K : 0;
    // A pair of steps is loaded into the registers of the one SETS before it as soon as that has been
    // multiplied; the first is issued before the rows are looked up (see glu_gemv_bf16_kernel; 8 tokens,
    // D 2048 / F 768: 50.3 -> 46.5 us for the pair of launches).
    u32x4 wq[SETS][2][M][4];
    uint32_t at = ((uint32_t)(wave * 16 + g * 4) * (uint32_t)N + lane_col) * 2u;  // as in glu_gemv_bf16_kernel
    auto load_pair = [&](int set) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int m = 0; m < M; ++m)
            wq[set][h][m][j] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc[m], at, j * N * 2, NT ? kNonTemporal : 0);
        at += (uint32_t)KSTEP * (uint32_t)N * 2u;
      }
    };
    if (DUAL) load_pair(0);
    __builtin_amdgcn_sched_barrier(0);
    // ---- the pass's rows -> LDS (rows past the expert's count as zeros) ---------------------------
    __syncthreads();  // the previous pass's sums have left LDS
    // (a row per group of threads, so that the row's place is looked up once and a thread's loads
    // are all in flight together; K is a multiple of 8 here: 16-byte pieces)
    {
      constexpr int TPR = THREADS / XR, INFLIGHT = DUAL ? 8 : 4;
      const int r = tid / TPR;
      const int c0 = tid - r * TPR;
      const int kchunks = K / 8;
      const bool has = r0 + r < cnt;
      // (the places of the rows of a wave, one or two, are uniform: scalar loads, which do not wait for
      // the vector ones)
      constexpr int RPW = XR / WAVES;
      size_t place[RPW];
      float weight[RPW];
#pragma unroll
      for (int i = 0; i < RPW; ++i) {
        const int rr = r0 + wave * RPW + i, row = off + (rr < cnt ? rr : 0);
        if constexpr (SELECT != 0) {
          const int t = selected_token(__builtin_amdgcn_readfirstlane(chosen.bits[e]), rr < cnt ? rr : 0);
          place[i] = (size_t)t * lda;
          weight[i] = row_w != nullptr ? selected_weight(chosen, t, e, sel.K) : 1.f;
          continue;
        }
        place[i] = (size_t)(row_map != nullptr ? row_map[row] : row) * lda;
        weight[i] = row_w != nullptr ? row_w[row] : 1.f;
      }
      const size_t src = RPW > 1 && lane >= 32 ? place[RPW - 1] : place[0];
      const float w = RPW > 1 && lane >= 32 ? weight[RPW - 1] : weight[0];
      u32x4 v[INFLIGHT];
      auto load_rows = [&](int cb) {
#pragma unroll
        for (int u = 0; u < INFLIGHT; ++u) {
          const int c = cb + u * TPR;
          v[u] = *reinterpret_cast<const u32x4*>(A + src + 8 * (c < kchunks ? c : 0));
        }
      };
      auto store_rows = [&](int cb) {
        if (row_w != nullptr) {  // (block-uniform; as dispatch's scaled copy rounds)
#pragma unroll
          for (int u = 0; u < INFLIGHT; ++u)
            v[u] = u32x4{scale_bf16x2(v[u][0], w), scale_bf16x2(v[u][1], w), scale_bf16x2(v[u][2], w),
                         scale_bf16x2(v[u][3], w)};
        }
#pragma unroll
        for (int u = 0; u < INFLIGHT; ++u) {
          const int c = cb + u * TPR;
          if (!has) v[u] = u32x4{0u, 0u, 0u, 0u};
          if (c >= kchunks) continue;
          u32x2* dst = reinterpret_cast<u32x2*>(xs + (size_t)r * ldx + 8 * c);  // 8-byte aligned
          dst[0] = u32x2{v[u][0], v[u][1]};
          dst[1] = u32x2{v[u][2], v[u][3]};
        }
      };
      load_rows(c0);
      // (behind the first of the rows, which are waited for first)
      __builtin_amdgcn_sched_barrier(0);
      if (!DUAL) load_pair(0);
      load_pair(1);
      __builtin_amdgcn_sched_barrier(0);
      store_rows(c0);
      for (int cb = c0 + TPR * INFLIGHT; cb < kchunks; cb += TPR * INFLIGHT) {
        load_rows(cb);
        store_rows(cb);
      }
    }
    if (tid < 4) xs[(size_t)XR * ldx + tid] = 0;
    lds_barrier();

    // ---- the stream over K --------------------------------------------------------------------------
    f32x4 acc[M][8];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int c = 0; c < 8; ++c) acc[m][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    int xk = wave * 16 + g * 4;  // the lane's first k of the next step
    auto multiply = [&](auto more) {  // (as in glu_gemv_bf16_kernel)
#pragma unroll
      for (int p = 0; p < SETS; ++p) {
        u32x2 xq[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          // (k rows past K, four together as K is a multiple of 4, meet zeros: chosen by address, a
          // select on the value would become a branch)
          xq[h] = *reinterpret_cast<const u32x2*>(xs + (xk < xend ? xrow + xk : xzero));
          xk += KSTEP;
        }
        const u32x4 xo = {xq[0][0], xq[0][1], xq[1][0], xq[1][1]};
        const bf16x8 xop = __builtin_bit_cast(bf16x8, xo);
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            // channel c of the lane: the low (c even) or high (c odd) half of dword c / 2 of each row
            const uint32_t sel = (c & 1) ? 0x07060302u : 0x05040100u;
            const u32x4(&a)[4] = wq[p][0][m];
            const u32x4(&b)[4] = wq[p][1][m];
            const u32x4 wo = {__builtin_amdgcn_perm(a[1][c >> 1], a[0][c >> 1], sel),
                              __builtin_amdgcn_perm(a[3][c >> 1], a[2][c >> 1], sel),
                              __builtin_amdgcn_perm(b[1][c >> 1], b[0][c >> 1], sel),
                              __builtin_amdgcn_perm(b[3][c >> 1], b[2][c >> 1], sel)};
            acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wo), xop,
                                                                 acc[m][c], 0, 0, 0);
            // (operands are formed four channels ahead at most: formed all at once they cost 64
            // registers and the kernel spills)
            if ((c & (DUAL ? 3 : 1)) == (DUAL ? 3 : 1)) __builtin_amdgcn_sched_barrier(0);
          }
        if constexpr (decltype(more)::value) {
          load_pair(p);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    for (int p0 = SETS; p0 < pairs; p0 += SETS) multiply(std::true_type{});
    multiply(std::false_type{});

    // ---- the waves' sums meet in LDS: (w + 4) onto w, then (w + 2) onto w, then 1 onto 0 ------------
    __syncthreads();  // every wave is done reading the rows: the sums take their place
#pragma unroll
    for (int half = 4; half >= 1; half >>= 1) {
      // (one address register per wave and constant offsets from it)
      if (wave >= half && wave < 2 * half) {
        float* rp = red + (wave - half) * (M * 32 * 64) + lane;
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
          for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) rp[(m * 32 + c * 4 + i) * 64] = acc[m][c][i];
      }
      __syncthreads();
      if (wave < half) {
        const float* rp = red + wave * (M * 32 * 64) + lane;
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
          for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[m][c][i] += rp[(m * 32 + c * 4 + i) * 64];
      }
      if (half > 1) __syncthreads();
    }
    // ---- wave 0: row m = l % 16, channels 8 (4 q + i) + c ---------------------------------------------
    if (wave == 0 && row_ok && r0 + c16 < cnt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = col_block * COLS + (4 * g + i) * 8;
        if (n >= N) continue;
        u32x4 o;
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          float v0 = acc[0][2 * h][i], v1 = acc[0][2 * h + 1][i];
          if (DUAL) {
            v0 = silu_f32(v0) * acc[M - 1][2 * h][i];
            v1 = silu_f32(v1) * acc[M - 1][2 * h + 1][i];
          }
          o[h] = (uint32_t)f32_to_bf16_bits(v0) | ((uint32_t)f32_to_bf16_bits(v1) << 16);
        }
        *reinterpret_cast<u32x4*>(C + (size_t)(off + r0 + c16) * ldc + n) = o;
      }
    }
  }
  }
}

}  // namespace fs2moe
