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
  int64_t rows_to_plan(int64_t bound) const { return counts != nullptr && planned > 0 ? planned : bound; }
};

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
// threads of the block must call it; the grid is a multiple of 8.  false: no tile for this block.
template <int BM, int THREADS>
__device__ __forceinline__ bool locate_tile_by_xcd(const Groups& g, int n_tiles, int& e, int& row0,
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
  __shared__ int s_wave[2][WAVES], s_found[4];
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
  return true;
}

}  // namespace fs2moe
