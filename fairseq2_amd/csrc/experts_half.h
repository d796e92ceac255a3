// Grouped GEMM on tiles of 128 x 128, 64 x 128, 64 x 64 or 64 x 256 (rows x "virtual" channels: gate and up channels of
// half as many each when DUAL), for launches whose 256 x 256 tiles (experts_dma.h, experts_mx.h) would leave CUs idle: bf16 rows
// against bf16 or e4m3 weights, block-scaled e4m3 rows against e4m3 weights.
//
// What bounds it: with few tiles a CU's time is its tiles' bytes over what it takes in.  Four waves bring a CU 47 GB/s
// through registers and 55 straight into LDS, eight 70 straight into LDS (every CU, blocks that do nothing else), so
// all eight waves load, straight into LDS, and the ring holds as many stages of 64 k as 136 KB allow (4, 5 or 8),
// all but one on their way.  80 rows, K 3200, N 1408: the throughput kernel's 6 tiles 42 us, 44 tiles of 64 x 64 19;
// 8 experts of 290 rows, K 5408, N 704: 89 us, 240 tiles of 64 x 128 45 us; on the fp8 pipe the layer at 3105 tokens,
// top-1 of 8 experts, D 768, F 8832 211 -> 167 us, with e4m3 weights and bf16 rows the layer at 146 tokens, top-6 of 32,
// D 1344, F 1536 124 -> 114.  Where there are several rounds of tiles the throughput kernels' cost the chip less
// (half_tiles::pick).
//
// The k order of every sum is the throughput kernels', on the same instructions: the same bits.
//
// In LDS a stage is its activations (rows of 128 bytes, 16-byte chunk kc of row r in place kc ^ ((r >> 1) & 7)) and
// its weights: (out, in) matrices like the activations; (in, out) matrices as rows of one k, of 256 bytes (chunk c of
// row k in place c ^ ((k & 3) << 2)) or 128 (c ^ (((k >> 1) & 1) << 2); with DUAL a sub-tile per matrix), so that the
// four rows a transposing read touches lie in different banks.  e4m3 tiles of 16 channels x 64 k lie as in memory,
// chunk c of channel r in place c ^ ((r >> 2) & 3), and become bf16 behind the read; against e4m3 rows a stage is 128 k,
// and weights lie like rows.
// Rows, channels and k that do not exist load zeros and touch no memory (buffer loads past the buffer's end).
//
// Blocks are persistent, one per CU; tile i of the list (expert-major, row block minor inside bands) goes to
// slot i % grid, where slots 32 c .. 32 c + 31 are the blocks of XCD c: what an XCD works on at a time are
// neighbours, which share weights and rows in its L2.  A block's tiles form one stream of stages.
#pragma once

#include <type_traits>

#include "common.h"
#include "experts_dma.h"
#include "experts_mx.h"
#include "tile_map.h"

namespace fs2moe {
namespace half_tiles {
constexpr int ROW_BYTES = 128;                 // of a row of activations in a stage: 64 k of bf16, 128 of e4m3
constexpr int WAVES = 8, THREADS = WAVES * 64;
constexpr int BAND = 8;                        // row blocks per band of the tile order
constexpr int LDE = 144, EPI_BYTES = WAVES * 16 * LDE;  // epilogue: 16 rows of up to 128 bytes per wave
constexpr int TABLE_INTS = 3 * FS2MOE_MAX_EXPERTS + 8;
// A fourth kind of weights next to FS2MOE_W_IN_OUT, FS2MOE_W_OUT_IN and dma::W_FP8_TILED (e4m3 codes against bf16
// rows): e4m3 codes against block-scaled e4m3 rows, on the fp8 matrix pipe (experts_mx.h).
constexpr int W_MX = 3;
// MX: the four block scales of every row of a stage, and what the waves that have none to load write
constexpr int ASCALE_BYTES = 512 + 256;
constexpr int weight_bytes(int BNV, int layout) { return BNV * (layout == dma::W_FP8_TILED ? 64 : ROW_BYTES); }
constexpr int stage_bytes(int BM, int BNV, int layout) {
  return BM * ROW_BYTES + weight_bytes(BNV, layout) + (layout == W_MX ? ASCALE_BYTES : 0);
}
// (as many as leave room for the epilogue and the tables, at most 8)
constexpr int stages(int BM, int BNV, int layout) {
  const int n = 136 * 1024 / stage_bytes(BM, BNV, layout);
  return n < 8 ? n : 8;
}
constexpr int smem_bytes(int BM, int BNV, int layout) {
  return stages(BM, BNV, layout) * stage_bytes(BM, BNV, layout) + EPI_BYTES + TABLE_INTS * 4;
}
// Up to how many rows an expert has on average the weights are loaded past the caches (twice as many: the same times).
// us without and with: 89 tokens, top-4 of 60, D 2048, F 1152 183, 171; 26, top-8 of 32, D 960, F 1536 99, 93; a training
// step of 494, top-1 of 16, D 2176, F 8320 1212, 1178.
inline int64_t once_rows(int BM) { return BM / 2; }
constexpr uint32_t NOWHERE = 0xfffffff0u;      // an offset past any buffer's end

// Gate/up of several rounds of tiles where no expert has more than 64 rows: tiles of 64 x 256, as many as the throughput
// kernel's and of the same weights, in pieces of rows as long (256 bytes).  A CU that takes weights for a few rows waits
// for memory: here two of three stages of 40 KB are on their way, loaded by every wave, there one unit of as much, loaded by four.
// Narrower tiles would fill more CUs, but their pieces of 128 bytes cost memory 10 % of its rate (64 tokens, top-6 of 64,
// D 4096, F 1024 281 -> 314 us).  Experts of more rows would have their weights read once for each row block (200 tokens of
// that layer by a popularity law 300 -> 335), and long sums stay where they were (40 tokens, top-1 of 16, D 5120, F 8192
// 674 -> 682).  us of the layer on the throughput kernel and on these, three layers and inputs in turn, evenly loaded and by
// a popularity law:
//   24 tokens, top-8 of 128, D 2048, F 768   194, 190; 83.4, 82.4      64       215, 212; 110.6, 106.9
//   48, top-4 of 60, D 1024, F 1408          110, 105; 58.1, 55.6      33, top-6 of 60, D 640, F 1600  86.5, 83.6; 49.6, 48.7
//   60, top-8 of 64, D 768, F 2048           131, 128; 79.6, 77.1      64, top-6 of 32, D 1280, F 704  66.5, 64.4; 68.7, 66.2
//   64, top-6 of 64, D 4096, F 1024          281, 282; 238, 238        20, top-2 of 8, D 4096, F 14336 497, 494; 480, 463
// (the last and 33 tokens: 64 x 128 by the model of rounds instead of the throughput kernel)
inline bool whole_rows(int most_rows, int K) { return most_rows >= 1 && most_rows <= 64 && K <= 4096; }

// Which of these tiles a launch takes: 0 none (the throughput kernel), else the smallest whose tiles are about
// one a CU: 1 64 x 64 (single products), 2 64 x 128, 3 128 x 128; 4 64 x 256 (whole_rows).
// us, throughput kernel and 1, 2, 3 (single products but for the last two, which are gate/up and down):
//   80 rows, K 3200, N 1408              42 against 19, 23, 28     (5, 44, 22, 11 tiles)
//   755 rows, K 1408, N 576              25 against 12, 14, 18
//   8 experts of 290, K 5408, N 704      89 against 59, 45, 56     (480, 240, 144 tiles: one round of the second)
//   3001 rows, K 1368, N 1024            28 against 27, 25, 20
//   16 experts of 375, K 1368, N 1024    33 against 62, 50, 37     (none fits one round)
//   32 of 35, D 1472, F 1216             90 against 79 (2), 80 (3) (the throughput kernel: 1.25 rounds)
//   64 of 23, D 2944, F 1840             377 against 394, 400      (memory)
// All are even loads.  Where a few rows reach a part of the experts, or most of the rows one, the tiles that count are
// few as well and these win by more.  So single products of bf16 take them on a smaller margin than a sixth, which codes
// need (they take longer to convert than the model's rounds say), us of the layer with that margin and with bf16's:
//   20 and 200 tokens, top-4 of 60 by a popularity law, D 1024, F 1408       60.3, 51.1; 73.0, 57.5
//   48 and 100, top-8 of 128 by one, D 2048, F 768                           96.2, 90.4; 130, 117
// Gate/up within 70 to 83 % of the model's time: evenly 11 % faster to 2 % slower on small tiles (24 shapes), by a
// popularity law 15 % faster to 18 % slower; within 85 to 88 % 1 % faster to 12 % slower at D 2048 and above.
// bf16: matrices and rows of bf16, not codes.  most: as for whole_rows.
inline int pick(bool dual, bool bf16, int64_t rows, int groups, int K, int N, int cus, int most = 0) {
  // Of the experts' rows only the device knows how they are spread: the planned ones (Groups), less what blocks of 16
  // pad them by, equally loaded.
  const int64_t real = rows > 15ll * groups ? rows - 15ll * groups : rows;
  const int64_t each = groups ? real / groups : real;
  auto tiles = [&](int bm, int bn) -> int64_t {
    const int64_t nt = (N + bn - 1) / bn;
    if (groups == 0) return (rows + bm - 1) / bm * nt;
    // (half of a last row block per expert)
    const int64_t blocks = groups + (each > bm / 2 ? (real - (int64_t)groups * (bm / 2)) / bm : 0);
    return (blocks < real ? blocks : real) * nt;
  };
  // (experts of many rows are not equally loaded: a few tiles more; of those of one row block some have none)
  const int64_t room = bf16 && each <= 32 ? cus : cus - cus / 16;
  if (bf16 && !dual && tiles(64, 64) <= room) return 1;
  if (tiles(64, dual ? 64 : 128) <= room) return 2;
  if (tiles(128, dual ? 64 : 128) <= room) return 3;
  if (dual && groups > 0 && whole_rows(most, K)) return 4;
  // Several rounds of tiles of a few rows: rounds of the throughput kernel (1 us per 64 k and 6 per tile, us) against
  // rounds of these (0.4 and 4), neither faster than memory delivers half of the experts' weights (5.2 TB/s; with few
  // tokens or a skewed load not all experts have rows), and a margin for what that leaves out.
  if (groups > 0 && each <= 64) {
    const int64_t units = (K + 63) / 64, active = groups < real ? groups : real;
    const int64_t memory = active * K * N * (dual ? 2 : 1) / 5200;  // ns
    auto rounds = [&](int64_t n) { return (n + cus - 1) / cus; };
    const int64_t whole = rounds(tiles(256, dual ? 128 : 256)) * (units * 1000 + 6000);
    const int64_t small = rounds(tiles(64, dual ? 64 : 128)) * (units * 400 + 4000);
    const int64_t percent = bf16 && !dual ? 100 - each / 4 : 83;
    if ((small > memory ? small : memory) * 100 < (whole > memory ? whole : memory) * percent) return 2;
  }
  return 0;
}
}  // namespace half_tiles

// 16 bytes per lane from a buffer to LDS, lane l's to lds + 16 l.  Written out because the compiler, which cannot
// tell the ring's stages apart, would wait for every load in flight before each LDS read.  The caller waits
// (vmcnt) in front of the barrier that hands the stage over.  BYTES 4: lane l's four to lds + 4 l.  PAST: past the
// caches (load_once).
// (m0 is named because the other kernels' loads to LDS set it as well; the compiler warns that it reserves it.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <int BYTES, bool PAST = false>
__device__ __forceinline__ void buffer_to_lds(const void* base, uint32_t off, uint32_t lds) {
  const uint64_t b = (uint64_t)base;
  const u32x4 rsrc = {(uint32_t)b, (uint32_t)(b >> 32) & 0xffffu, half_tiles::NOWHERE, 0x00020000u};
  if constexpr (BYTES == 16 && PAST)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen nt lds" ::"v"(off), "s"(rsrc),
                 "s"(lds)
                 : "memory", "m0");
  else if constexpr (BYTES == 16)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off), "s"(rsrc),
                 "s"(lds)
                 : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dword %0, %1, 0 offen lds" ::"v"(off), "s"(rsrc),
                 "s"(lds)
                 : "memory", "m0");
}
#pragma clang diagnostic pop

// The block-scaled e4m3 kernels' further operands: scale bytes of the rows in and (gate/up) out, k-group major
// ([K / 128][rows][4]), and how many rows each array has.
struct HalfMx {
  const uint8_t* As;
  uint8_t* Cs;
  int a_rows, c_rows;
};

// Arguments as glu_gemm_bf16_dma_kernel takes them (KEEP_GU: the products' destinations in S0 and S1; TWO_SRC:
// the second activations in S0, the second weights in B1), or for W_MX as glu_gemm_mx_kernel does.  n_tiles: of 64
// (DUAL) or 128 channels.
// ONCE: the weights are loaded past the caches, for launches most of whose experts have one row block.
template <int BM, int BNV, bool DUAL, int BLAYOUT, bool KEEP_GU = false, bool TWO_SRC = false, bool ONCE = false>
__global__ __launch_bounds__(half_tiles::THREADS, 2) void glu_gemm_half_kernel(
    const uint8_t* __restrict__ A, const int32_t* __restrict__ row_map, int lda,
    const uint8_t* __restrict__ B0, const uint8_t* __restrict__ B1, const float* __restrict__ S0,
    const float* __restrict__ S1, uint8_t* __restrict__ C, int ldc, int Kdim, int N, Groups g, int n_tiles,
    HalfMx mxa) {
  using namespace half_tiles;
  constexpr bool KN = BLAYOUT == FS2MOE_W_IN_OUT, FP8 = BLAYOUT == dma::W_FP8_TILED, MX = BLAYOUT == W_MX;
  constexpr bool CODES = FP8 || MX;        // weights as e4m3 tiles with channel scales S0, S1
  static_assert(!KEEP_GU || (DUAL && !CODES), "the products are kept by the bf16 gate/up kernel only");
  static_assert(!TWO_SRC || (!DUAL && !CODES), "two sources: one bf16 matrix each");
  static_assert((BM == 64 || BM == 128) && (BNV == 128 || (BNV == 64 && !DUAL && !CODES) ||
                                            (BNV == 256 && BM == 64 && DUAL && !CODES)),
                "tiles that the loads are cut for");
  constexpr int A_BYTES = BM * ROW_BYTES, B_BYTES = weight_bytes(BNV, BLAYOUT);
  constexpr int STAGE_BYTES = stage_bytes(BM, BNV, BLAYOUT);
  constexpr int STAGES = stages(BM, BNV, BLAYOUT), RING_BYTES = STAGES * STAGE_BYTES;
  constexpr int KU = MX ? 128 : 64;              // k per stage
  constexpr int ASIZE = MX ? 1 : 2, WSIZE = CODES ? 1 : 2;  // bytes of an element
  constexpr int SLICES = MX ? 2 : 4;             // of a stage's k, each an instruction per fragment
  constexpr int PA = BM / 64, PB = FP8 ? 1 : BNV / 64, LOADS = PA + PB + (MX ? 1 : 0);  // of a wave and stage
  constexpr int BN = DUAL ? BNV / 2 : BNV;       // real channels per tile
  constexpr int BROW = BN * 2;                   // bytes per LDS row of (in, out) weights
  constexpr int NF = DUAL || BM * BNV == 128 * 128 ? 2 : 1;  // 32-channel fragments of a wave
  constexpr int WN = BNV / 32 / NF;              // waves across the channels
  constexpr int COLS = DUAL ? 32 : NF * 32;      // channels a wave writes
  constexpr int TILE_STORES = MX && DUAL ? 2 : COLS / 16 * (KEEP_GU ? 3 : 1);  // of a wave
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem_raw[];
  int32_t* s_start = reinterpret_cast<int32_t*>(smem_raw + RING_BYTES + EPI_BYTES);  // [E + 1] row blocks
  int32_t* s_counts = s_start + FS2MOE_MAX_EXPERTS + 4;
  int32_t* s_offsets = s_counts + FS2MOE_MAX_EXPERTS;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // The wave's 32 rows and its share of the channels; waves past the tile only load.  (Waves w and w + 4 share a
  // SIMD.)
  const int wm = wave / WN, wn = wave % WN;
  const int lr = lane & 31, lk = lane >> 5;

  // ---- row blocks of the experts before each
  const bool dense = g.counts == nullptr;
  const int E = dense ? 1 : g.E;
  {
    __shared__ int s_wave_tot[WAVES];
    const int cnt = dense ? (tid == 0 ? g.dense_rows : 0) : (tid < E ? g.counts[tid] : 0);
    const int off = dense || tid >= E ? 0 : g.offsets[tid];
    const int blocks = (cnt + BM - 1) / BM;
    int incl = blocks;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, kWave);
      if (lane >= o) incl += v;
    }
    if (lane == 63) s_wave_tot[wave] = incl;
    __syncthreads();
    int base = 0;
    for (int w = 0; w < wave; ++w) base += s_wave_tot[w];
    if (tid < E) {
      s_start[tid] = base + incl - blocks;
      s_counts[tid] = cnt;
      s_offsets[tid] = off;
    }
    if (tid == E - 1) s_start[E] = base + incl;
    __syncthreads();
  }
  const int slot = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3), grid = (int)gridDim.x;
  const int tiles = s_start[E] * n_tiles;  // (the host guarantees that it fits 31 bits)
  const int my_tiles = slot < tiles ? (tiles - slot + grid - 1) / grid : 0;
  if (my_tiles == 0) return;
  const int units = (Kdim + KU - 1) / KU, nu = (TWO_SRC ? 2 : 1) * units;  // stages per tile

  struct Tile {
    int e, row0, row_end, n0;
  };
  auto locate = [&](int j) {
    const int t = slot + j * grid, mt = t / n_tiles;  // mt: which expert, as its tiles are contiguous
    int found = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + lane;
      const unsigned long long m = __ballot(e < E && s_start[e] <= mt && mt < s_start[e + 1]);
      if (m) found = e0 + (int)__builtin_ctzll(m);
    }
    found = __builtin_amdgcn_readfirstlane(found);
    const int first = s_start[found], l = t - first * n_tiles, per_band = BAND * n_tiles;
    const int b = l / per_band, i = l - b * per_band;
    const int left = s_start[found + 1] - first - b * BAND, high = left < BAND ? left : BAND;
    const int nt = i / high, row = (b * BAND + i - nt * high) * BM, cnt = s_counts[found];
    Tile r;
    r.e = found;
    r.row0 = __builtin_amdgcn_readfirstlane(s_offsets[found] + row);
    r.row_end = __builtin_amdgcn_readfirstlane(s_offsets[found] + (cnt < row + BM ? cnt : row + BM));
    r.n0 = __builtin_amdgcn_readfirstlane(nt) * BN;
    return r;
  };
  const size_t wstride = (size_t)Kdim * N * WSIZE;  // bytes of one expert's matrix

  // ---- the stream of stages into LDS: stage u of the block goes to slot u % STAGES
  const uint32_t ring = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem_raw;
  // The wave's pieces of 1 KB: rows 8 wave .. 8 wave + 7 of the activations and, 64 further on, 8 more; of the
  // weights likewise (with DUAL the first half of them of the gate, the second of the up matrix).  A lane's place in piece i:
  uint32_t pa[PA], pb[PB];
  // chunk of the row's 128 bytes that the lane fetches (the same for both pieces), of activations and (out, in)
  // weights; k row of (in, out) weights in the stage
  const int kc = (lane & 7) ^ ((4 * wave + (lane >> 4)) & 7);
  constexpr int KROWS = 1024 / BROW, KCHUNKS = BROW / 16;  // rows and chunks of a piece of (in, out) weights
  // (piece i is the wave's i % PM-th of matrix i / PM)
  constexpr int PM = DUAL && !FP8 ? PB / 2 : PB;
  auto piece = [&](int i) { return wave + 8 * (i % PM); };
  auto k_key = [](int k) { return BROW == 128 ? ((k >> 1) & 1) << 2 : (k & 3) << 2; };
  int ld_tile = 0, ld_ku = 0, ld_slot = 0;
  const uint8_t* ld_b[2] = {B0, B0};
  const uint8_t* ld_as = mxa.As;
  uint32_t pas = 0;  // MX: the lane's row of scales
  auto setup_tile = [&]() {
    const Tile t = locate(ld_tile);
    ld_b[0] = B0 + (size_t)t.e * wstride;
    ld_b[1] = DUAL || TWO_SRC ? B1 + (size_t)t.e * wstride : ld_b[0];
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      const int piece_row = 8 * (wave + 8 * i);  // uniform
      int row = t.row0 + piece_row + (lane >> 3);
      const bool in = row < t.row_end;
      if (row_map != nullptr) {
        // (scalar loads: a vector load would be waited for with every stage in flight; rows past the end
        // repeat the last one's entry)
        int entry[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const int at = t.row0 + piece_row + r;
          entry[r] = row_map[at < t.row_end ? at : t.row_end - 1];
        }
        row = entry[0];
#pragma unroll
        for (int r = 1; r < 8; ++r) row = lane >> 3 == r ? entry[r] : row;
      }
      pa[i] = in ? (uint32_t)row * (uint32_t)lda * ASIZE + (uint32_t)kc * 16u : NOWHERE;
    }
    if constexpr (MX) {
      // waves 0 .. BM / 64 - 1 load the scales of 64 rows each
      const int at = t.row0 + 64 * wave + lane;
      const bool in = wave < BM / 64 && at < t.row_end;
      pas = NOWHERE;
      if (wave < BM / 64) pas = in ? (uint32_t)(row_map != nullptr ? row_map[at] : at) * 4u : NOWHERE;
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      if constexpr (CODES) {
        // tiles of 16 channels x 64 k, 1 KB each, [channel / 16][k / 64]
        const int nkb = Kdim / 64;
        if constexpr (FP8) {
          // a piece is a tile: the lane's chunk of 16 k of channel lane / 4, chunk c of channel r in place
          // c ^ ((r >> 2) & 3)
          const int r = lane >> 2, c = (lane & 3) ^ ((r >> 2) & 3);
          const int group = t.n0 / 16 + (DUAL ? wave & 3 : wave);
          pb[i] = group < N / 16 ? (uint32_t)group * (uint32_t)nkb * 1024u + (uint32_t)(r * 64 + c * 16) : NOWHERE;
        } else {
          // a piece is 8 channel rows of 128 k, from two tiles
          const int P = piece(i), r = 8 * (P & 1) + (lane >> 3);
          const int group = t.n0 / 16 + (P >> 1);
          pb[i] = group < N / 16 ? ((uint32_t)group * (uint32_t)nkb + (uint32_t)(kc >> 2)) * 1024u +
                                       (uint32_t)(r * 64 + (kc & 3) * 16)
                                 : NOWHERE;
        }
      } else if constexpr (KN) {
        const int k = KROWS * piece(i) + lane / KCHUNKS, key = k_key(k);
        const int col = t.n0 + ((lane % KCHUNKS) ^ key) * 8;
        pb[i] = col < N ? ((uint32_t)k * (uint32_t)N + (uint32_t)col) * 2u : NOWHERE;
      } else {
        const int ch = t.n0 + 8 * piece(i) + (lane >> 3);
        pb[i] = ch < N ? (uint32_t)ch * (uint32_t)Kdim * 2u + (uint32_t)kc * 16u : NOWHERE;
      }
    }
  };
  // Load l of the stage to load next: the activations' pieces, the weights', the rows' scales.
  auto load = [&](int l) {
    const bool of_a = l < PA, of_scales = l == PA + PB;
    const int i = of_a ? l : l - PA;
    const bool second = TWO_SRC && ld_ku >= units;
    const int ku = second ? ld_ku - units : ld_ku;
    // (behind the last tile nothing is left)
    const int left = ld_tile < my_tiles ? Kdim - ku * KU : 0;
    const uint32_t stage = ring + (uint32_t)(ld_slot * STAGE_BYTES);
    const uint32_t at = stage + (uint32_t)((of_a ? 0 : A_BYTES) + (wave + 8 * i) * 1024);
    if (of_scales) {
      const uint32_t to = stage + (uint32_t)(A_BYTES + B_BYTES + (wave < BM / 64 ? wave * 256 : 512));
      buffer_to_lds<4>(ld_as + (size_t)ku * (size_t)mxa.a_rows * 4, left > 0 ? pas : NOWHERE, to);
    } else if (of_a) {
      const uint8_t* src = second ? reinterpret_cast<const uint8_t*>(S0) : A;
      buffer_to_lds<16>(src + (size_t)ku * ROW_BYTES, kc * (16 / ASIZE) < left ? pa[i] : NOWHERE, at);
    } else {
      const uint8_t* src = TWO_SRC ? ld_b[second ? 1 : 0] : ld_b[DUAL ? (FP8 ? wave >> 2 : i / PM) : 0];
      if constexpr (FP8) {
        buffer_to_lds<16, ONCE>(src + (size_t)ku * 1024, left > 0 ? pb[i] : NOWHERE, at);
      } else if constexpr (MX) {
        buffer_to_lds<16, ONCE>(src + (size_t)ku * 2048, left > 0 ? pb[i] : NOWHERE, at);
      } else if constexpr (KN) {
        const int k = KROWS * piece(i) + lane / KCHUNKS;
        buffer_to_lds<16, ONCE>(src + (size_t)ku * KU * N * 2, k < left ? pb[i] : NOWHERE, at);
      } else {
        buffer_to_lds<16, ONCE>(src + (size_t)ku * ROW_BYTES, kc * 8 < left ? pb[i] : NOWHERE, at);
      }
    }
  };
  auto loaded = [&]() {
    ld_slot = ld_slot + 1 == STAGES ? 0 : ld_slot + 1;
    if (++ld_ku == nu) {
      ld_ku = 0;
      if (++ld_tile < my_tiles) setup_tile();
    }
  };

  // ---- fragments (bytes from the start of a stage)
  const int xrow = (wm * 32 + lr) * 128, xkey = (lr >> 1) & 7;
  int wb[NF];
#pragma unroll
  for (int fn = 0; fn < NF; ++fn) {
    const int ch = wn * COLS + (DUAL ? fn * BN : fn * 32) + lr;  // virtual channel
    if constexpr (KN) {
      const int s = lane & 15, k = lk * 8 + (s >> 2);
      const int col = wn * COLS + (DUAL ? 0 : fn * 32) + ((lane >> 4) & 1) * 16 + (s & 3) * 4;
      wb[fn] = A_BYTES + (DUAL ? fn * (B_BYTES / 2) : 0) + k * BROW + (((col >> 3) ^ k_key(k)) * 16) + (col & 7) * 2;
    } else if constexpr (FP8) {
      wb[fn] = A_BYTES + (ch >> 4) * 1024 + (ch & 15) * 64 + lk * 8;
    } else {
      wb[fn] = A_BYTES + ch * 128;
    }
  }
  typedef __attribute__((ext_vector_type(8))) int i32x8;
  struct Frags {
    std::conditional_t<MX, i32x8, bf16x8> x;
    std::conditional_t<MX, i32x8, std::conditional_t<FP8, u32x2, bf16x8>> w[NF];
  };
  auto read = [&](Frags& f, int at_slot, int ks) {
    const uint8_t* st = smem_raw + at_slot * STAGE_BYTES;
    if constexpr (MX) {
      // (the operand's bytes: k 16 lk .. and k 32 + 16 lk .. of the slice's 64, see experts_mx.h)
      const int o0 = ((4 * ks + lk) ^ xkey) * 16, o1 = ((4 * ks + 2 + lk) ^ xkey) * 16;
      auto read32 = [&](const uint8_t* row) {
        const u32x4 lo = *reinterpret_cast<const u32x4*>(row + o0), hi = *reinterpret_cast<const u32x4*>(row + o1);
        return i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
      };
      f.x = read32(st + xrow);
#pragma unroll
      for (int fn = 0; fn < NF; ++fn) f.w[fn] = read32(st + wb[fn]);
    } else {
      const int xo = ((2 * ks + lk) ^ xkey) * 16;
      f.x = lds_read_frag(reinterpret_cast<const uint16_t*>(st + xrow + xo));
#pragma unroll
      for (int fn = 0; fn < NF; ++fn) {
        if constexpr (KN)
          f.w[fn] = lds_read_frag_tr(reinterpret_cast<const uint16_t*>(st + wb[fn] + ks * 16 * BROW),
                                     reinterpret_cast<const uint16_t*>(st + wb[fn] + ks * 16 * BROW + 4 * BROW));
        else if constexpr (FP8)
          f.w[fn] = *reinterpret_cast<const u32x2*>(st + wb[fn] + ((ks ^ ((lr >> 2) & 3)) * 16));
        else
          f.w[fn] = lds_read_frag(reinterpret_cast<const uint16_t*>(st + wb[fn] + xo));
      }
    }
  };
  f32x16 acc[NF];
  int row_scales = 0;  // MX: the stage's four block scales of the lane's row, from its half wave's first on
  auto multiply = [&](const Frags& f, auto slice) {
    (void)slice;
#pragma unroll
    for (int fn = 0; fn < NF; ++fn) {
      if constexpr (MX)  // (weights: scale 1; the row's scale of block 2 slice + lk)
        acc[fn] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f.w[fn], f.x, acc[fn], 0, 0, 0, 0x7f7f7f7f,
                                                                   decltype(slice)::value == 0 ? 0 : 2, row_scales);
      else if constexpr (FP8)
        acc[fn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fp8x8_to_bf16x8(f.w[fn][0], f.w[fn][1]), f.x, acc[fn], 0, 0, 0);
      else
        acc[fn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.w[fn], f.x, acc[fn], 0, 0, 0);
    }
  };
  // CODES: the scales of the lane's channels 8 q + 4 lk + {0..3} of fragment fn
  f32x4 wscale[CODES ? NF : 1][4];
  auto load_wscales = [&](const Tile& t) {
#pragma unroll
    for (int fn = 0; fn < NF; ++fn)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int ch = t.n0 + wn * COLS + (DUAL ? 0 : fn * 32) + 8 * q + 4 * lk;
        const float* sc = DUAL && fn == 1 ? S1 : S0;
        wscale[CODES ? fn : 0][q] = *reinterpret_cast<const f32x4*>(sc + (size_t)t.e * N + (ch < N ? ch : 0));
      }
  };

  // ---- epilogue: through the wave's own piece of LDS, so that a store instruction writes whole pieces of rows.
  // 16 rows at a time of COLS columns, 144 bytes apart.  Every store is issued (what does
  // not exist with an offset past the buffer's end): the stages' waits count them.
  auto store_rows = [&](uint16_t* out, const Tile& t, auto value) {
    constexpr int LPR = COLS / 8, ROWS = 64 / LPR;  // lanes per row, rows per store
    uint8_t* buf = smem_raw + RING_BYTES + wave * 16 * LDE;
    const int r_lane = lane / LPR, n = wn * COLS + (lane % LPR) * 8;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        out + (size_t)t.row0 * ldc + t.n0, 0, NOWHERE, 0x00020000);  // (ldc: elements)
    u32x2 o[COLS / 32][4];
#pragma unroll
    for (int fn = 0; fn < COLS / 32; ++fn)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = value(fn, 4 * q + j);
        o[fn][q] = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (lr >> 4 == h) {
#pragma unroll
        for (int fn = 0; fn < COLS / 32; ++fn)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<u32x2*>(buf + (lr & 15) * LDE + (fn * 32 + 8 * q + 4 * lk) * 2) = o[fn][q];
      }
      // (the wave's LDS traffic runs in order: only the compiler has to keep it)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int p = 0; p < 16 / ROWS; ++p) {
        const int row = p * ROWS + r_lane, m = wm * 32 + h * 16 + row;
        const u32x4 v = *reinterpret_cast<const u32x4*>(buf + row * LDE + (lane % LPR) * 16);
        uint32_t at = ((m < BM) & (t.row0 + m < t.row_end) & (t.n0 + n < N)) ? (uint32_t)(m * ldc + n) * 2u : NOWHERE;
        asm volatile("" : "+v"(at));  // (chosen before the store, not by a branch around it)
        __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, at, 0, 0);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  };

  // MX, DUAL: the gated product as e4m3 codes with a scale byte per row and 32 channels (the wave's).
  auto store_codes = [&](const Tile& t) {
    uint8_t* buf = smem_raw + RING_BYTES + wave * 16 * LDE;  // 32 rows of 32 bytes
    float v[16], amax = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      v[i] = silu_f32(acc[0][i] * wscale[0][i >> 2][i & 3]) * (acc[NF - 1][i] * wscale[CODES ? NF - 1 : 0][i >> 2][i & 3]);
      amax = fmaxf(amax, fabsf(v[i]));
    }
    // (the other half of the block sits in lane ^ 32)
    amax = fmaxf(amax, __int_as_float(__builtin_amdgcn_ds_bpermute((lane ^ 32) << 2, __float_as_int(amax))));
    const int X = mx::block_exponent(amax);
    const float inv = __builtin_ldexpf(1.0f, -X);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<uint32_t*>(buf + lr * 32 + q * 8 + lk * 4) =
          mx::to_e4m3x4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3], inv);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int n = wn * 32, r = lane >> 1, m = wm * 32;
    const u32x4 codes = *reinterpret_cast<const u32x4*>(buf + lane * 16);
    const __amdgpu_buffer_rsrc_t c_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(C + (size_t)t.row0 * ldc + t.n0, 0, NOWHERE, 0x00020000);
    uint32_t at = ((m < BM) & (t.row0 + m + r < t.row_end) & (t.n0 + n < N))
                      ? (uint32_t)((m + r) * ldc + n + (lane & 1) * 16) : NOWHERE;
    asm volatile("" : "+v"(at));
    __builtin_amdgcn_raw_buffer_store_b128(codes, c_rsrc, at, 0, 0);
    const int block = (t.n0 + n) >> 5;
    const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        mxa.Cs + ((size_t)(block >> 2) * mxa.c_rows + t.row0) * 4 + (block & 3), 0, NOWHERE, 0x00020000);
    at = ((m < BM) & (lk == 0) & (t.row0 + m + lr < t.row_end) & (t.n0 + n < N)) ? (uint32_t)(m + lr) * 4u : NOWHERE;
    asm volatile("" : "+v"(at));
    __builtin_amdgcn_raw_buffer_store_b8((uint8_t)(X + 127), s_rsrc, at, 0, 0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };

  setup_tile();
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) {
#pragma unroll
    for (int l = 0; l < LOADS; ++l) load(l);
    loaded();
  }
  // How many of the stages to wait for were asked for in front of the last tile's stores: what was issued
  // behind them need not have completed, the stores neither (loads and stores complete in order of issue).
  int before_stores = 0, at_slot = 0;
  for (int j = 0; j < my_tiles; ++j) {
    const Tile t = locate(j);
    const bool active = wm * 32 < BM && t.row0 + wm * 32 < t.row_end;
#pragma unroll
    for (int fn = 0; fn < NF; ++fn)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[fn][i] = 0.f;
    if constexpr (CODES) load_wscales(t);
    for (int ku = 0; ku < nu; ++ku) {
      // this wave's part of the stage, the oldest on its way, has to be there
      if (before_stores > 0) {
        --before_stores;
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 2) * LOADS + TILE_STORES) : "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 2) * LOADS) : "memory");
      }
      lds_barrier();  // and the stage before has been read by everyone: its slot takes the next one to load
      // (a load takes a wave its turn among the eight: they go out between the products)
      if (active) {
        Frags f[2];
        read(f[0], at_slot, 0);
        read(f[1], at_slot, 1);
        if constexpr (MX)
          row_scales = (int)(*reinterpret_cast<const uint32_t*>(smem_raw + at_slot * STAGE_BYTES + A_BYTES + B_BYTES +
                                                                (wm * 32 + lr) * 4) >> (8 * lk));
        __builtin_amdgcn_sched_barrier(0);
        auto slice = [&](auto ks_c) {
          constexpr int ks = decltype(ks_c)::value;
#pragma unroll
          for (int l = ks * LOADS / SLICES; l < (ks + 1) * LOADS / SLICES; ++l) load(l);
          __builtin_amdgcn_sched_barrier(0);
          multiply(f[ks & 1], ks_c);
          if constexpr (ks + 2 < SLICES) read(f[ks & 1], at_slot, ks + 2);
          __builtin_amdgcn_sched_barrier(0);
        };
        slice(std::integral_constant<int, 0>{});
        slice(std::integral_constant<int, 1>{});
        if constexpr (SLICES == 4) {
          slice(std::integral_constant<int, 2>{});
          slice(std::integral_constant<int, 3>{});
        }
      } else {
#pragma unroll
        for (int l = 0; l < LOADS; ++l) load(l);
      }
      loaded();
      at_slot = at_slot + 1 == STAGES ? 0 : at_slot + 1;
    }
    before_stores = STAGES - 1;
    if constexpr (KEEP_GU) {
      store_rows(reinterpret_cast<uint16_t*>(const_cast<float*>(S0)), t, [&](int, int i) { return acc[0][i]; });
      store_rows(reinterpret_cast<uint16_t*>(const_cast<float*>(S1)), t, [&](int, int i) { return acc[NF - 1][i]; });
    }
    if constexpr (MX && DUAL) {
      store_codes(t);
    } else {
      store_rows(reinterpret_cast<uint16_t*>(C), t, [&](int fn, int i) {
        if constexpr (CODES && DUAL)
          return silu_f32(acc[0][i] * wscale[0][i >> 2][i & 3]) * (acc[NF - 1][i] * wscale[NF - 1][i >> 2][i & 3]);
        else if constexpr (CODES)
          return acc[fn][i] * wscale[fn][i >> 2][i & 3];
        else
          return DUAL ? silu_f32(acc[0][i]) * acc[NF - 1][i] : acc[fn][i];
      });
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may arrive in LDS after the block
}

}  // namespace fs2moe
