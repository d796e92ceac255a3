// Output-tile scheduling of the grouped GEMMs: which expert and row range a block works on.
#pragma once

#include "common.h"

namespace fs2moe {

struct Groups {
  const int32_t* counts;   // [E] tokens per expert, or nullptr for one dense group
  const int32_t* offsets;  // [E + 1] first row of each expert
  int E;
  int dense_rows;
  // host: the planned rows (common.h) where the caller knows them, else 0 and the buffers' size stands for them; the
  // choice of tiles goes by them, while grids and addresses go by the buffers
  int planned = 0;
  // host: whether the launch may load its weights past the caches (load_once); it does where few rows an expert make
  // most tiles their expert's only row block
  int once_past_cache = 0;
  // host: how many rows an expert has at most, where the caller knows it (0: it does not)
  int most = 0;
  int64_t rows_to_plan(int64_t bound) const { return counts != nullptr && planned > 0 ? planned : bound; }
};

// Whether the weights that a call's `pairs` rows can reach, each row an expert of its own, are more than the last-level
// cache (256 MB) holds: what is read once is then loaded past the caches, where otherwise some of it may still lie there
// from the call before.  A skewed load reaches fewer, and its weights may fit: that costs a call 3 % whose own weights
// still lie there, and gives 17 % to one with other layers' calls in between.  D 2048, F 768, 128 experts, top-8 (9.4 MB an
// expert), us of the layer under a graph without and with the hint, on the same input again, on 24 inputs in turn, and with
// 1.3 GB of other memory read and written in between:
//   1 token (75 MB at most)                                44.1, 46.8    48.2, 47.8    61.2, 55.3
//   4, by a popularity law (302 MB at most)                59.9, 61.2    63.2, 64.4    83.0, 69.4
//   8 by one (604 at most, 210)                            71.2, 73.5    72.0, 73.9    98.7, 81.4
//   8 evenly (470)                                        140.0, 128.7  139.2, 129.1  170.0, 135.8
//   16 by a law                                            80.6, 80.7    80.4, 81.0   110.5, 87.2
// 64 tokens by a law with e4m3 weights (without a graph)   63.3, 67.5    62.0, 67.1    82.7, 71.1
// (What fits even so, up to 320 MB, is left in the caches: a program of one layer.)
// Whole layers of 262 MB, by a popularity law, which leaves some experts out: 60 of D 704, F 1088, 720 tokens 66.0, 69.5;
// of 288 MB 62.9, 64.5 (128 of D 768, F 512), 86.8, 84.3 (64 of D 1024, F 768); of 432 MB 125, 121.  One group, the
// shared expert, counts for more: the routed ones' weights go by beside it.
inline bool weights_past_cache(int groups, int64_t pairs, int64_t D, int64_t F, int weight_bytes) {
  const int64_t reached = groups == 0 ? 1 : pairs < groups ? pairs : groups;
  return reached * 3 * D * F * weight_bytes > (groups == 0 ? 128ll << 20 : 320ll << 20);
}
// (the rows of experts that are not planned: as many as the buffers hold)
inline int64_t pairs_of(const Groups& g, int64_t rows_bound) {
  return g.counts != nullptr && g.planned > 15ll * g.E ? g.planned - 15ll * g.E : rows_bound;
}

// Up to how many rows an expert has on average most tiles of 256 rows are their expert's only row block (launch_dma has
// the times).
constexpr int64_t kOnceRows = 128, kOnceRowsTraining = 192;

// Finds the (expert, row range) of m-tile `mt`.  All 256 threads of the block must call it.
template <int BM>
__device__ __forceinline__ bool locate_tile(const Groups& g, int mt, int& e, int& row0,
                                            int& row_end) {
  if (g.counts == nullptr) {
    e = 0;
    row0 = mt * BM;
    row_end = g.dense_rows;
    return row0 < row_end;
  }
  __shared__ int s_wave_tot[2][4];
  __shared__ int s_tile[3];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid == 0) s_tile[0] = -1;
  // the experts 256 at a time (one per thread), carrying the tiles of the rounds before
  int carried = 0;
  for (int e0 = 0; e0 < g.E; e0 += 256) {
    const int ex = e0 + tid, par = (e0 >> 8) & 1;
    const int cnt = ex < g.E ? g.counts[ex] : 0;
    const int tiles = (cnt + BM - 1) / BM;
    int incl = tiles;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      int v = __shfl_up(incl, off, kWave);
      if (lane >= off) incl += v;
    }
    if (lane == 63) s_wave_tot[par][wave] = incl;
    __syncthreads();
    int base = carried;
    for (int w = 0; w < wave; ++w) base += s_wave_tot[par][w];
    const int excl = base + incl - tiles;
    if (tiles > 0 && mt >= excl && mt < excl + tiles) {
      const int off = g.offsets[ex];
      s_tile[0] = ex;
      s_tile[1] = off + (mt - excl) * BM;
      s_tile[2] = off + cnt;
    }
    for (int w = 0; w < 4; ++w) carried += s_wave_tot[par][w];
  }
  __syncthreads();
  e = s_tile[0];
  row0 = s_tile[1];
  row_end = s_tile[2];
  return e >= 0;
}

// The tile of block blockIdx.x when the grid's tiles (m-tiles of BM rows x n_tiles, channel block minor)
// are cut into eight runs of neighbours, one per XCD (block b runs on XCD b % 8, each with its own L2):
// the blocks an XCD holds at a time then share their rows and their expert's weights.  All THREADS
// threads of the block must call it; the grid is a multiple of 8.  scratch: 4 + THREADS / 32 words of LDS, free again
// afterwards.  false: no tile for this block.
template <int BM, int THREADS>
__device__ __forceinline__ bool locate_tile_by_xcd(const Groups& g, int n_tiles, int32_t* scratch, int& e, int& row0,
                                                   int& row_end, int& nt) {
  const int idx = blockIdx.x >> 3, xcd = blockIdx.x & 7;
  if (g.counts == nullptr) {
    const int total = (g.dense_rows + BM - 1) / BM * n_tiles, per = (total + 7) / 8;
    const int t = xcd * per + idx;
    if (idx >= per || t >= total) return false;
    e = 0;
    nt = t % n_tiles;
    row0 = t / n_tiles * BM;
    row_end = g.dense_rows;
    return true;
  }
  constexpr int ROUNDS = FS2MOE_MAX_EXPERTS / THREADS, WAVES = THREADS / 64;
  int32_t* s_found = scratch;
  int32_t(*s_wave)[WAVES] = reinterpret_cast<int32_t(*)[WAVES]>(scratch + 4);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // tiles in all, then the one of this block (the experts one per thread)
  int cnt[ROUNDS], excl[ROUNDS], carried = 0;
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    cnt[r] = excl[r] = 0;
    if (r * THREADS >= g.E) continue;  // block-uniform
    const int ex = r * THREADS + tid;
    cnt[r] = ex < g.E ? g.counts[ex] : 0;
    const int tiles = (cnt[r] + BM - 1) / BM;
    int incl = tiles;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(incl, off, kWave);
      if (lane >= off) incl += v;
    }
    if (lane == 63) s_wave[r & 1][wave] = incl;
    __syncthreads();
    int base = carried;
    for (int w = 0; w < wave; ++w) base += s_wave[r & 1][w];
    excl[r] = base + incl - tiles;
    for (int w = 0; w < WAVES; ++w) carried += s_wave[r & 1][w];
  }
  const int total = carried * n_tiles, per = (total + 7) / 8, t = xcd * per + idx;
  if (idx >= per || t >= total) return false;  // block-uniform
  const int mt = t / n_tiles;
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int tiles = (cnt[r] + BM - 1) / BM;
    if (tiles > 0 && mt >= excl[r] && mt < excl[r] + tiles) {
      const int off = g.offsets[r * THREADS + tid];
      s_found[0] = r * THREADS + tid;
      s_found[1] = off + (mt - excl[r]) * BM;
      s_found[2] = off + cnt[r];
    }
  }
  __syncthreads();
  e = s_found[0];
  row0 = s_found[1];
  row_end = s_found[2];
  nt = t - mt * n_tiles;
  __syncthreads();  // (scratch has been read)
  return true;
}

}  // namespace fs2moe
