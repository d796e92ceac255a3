// Backward pass of the MoE feed-forward layer: the kernels that the forward pass has no use for.
//
// The gradient of out = sum_k w_k * expert_k(x) [+ shared(x)] reuses the forward machinery wherever the
// operation is the same with other operands (a grouped GEMM against the transposed weights is the
// grouped GEMM in the other weight orientation; the gather of output gradients into expert order is
// dispatch; the scatter of input gradients back to token order is combine).  What is new:
//   * grouped_wgrad_kernel   dW_e = A_e^T B_e, a GEMM whose contraction runs over the expert's rows
//   * swiglu_backward_kernel element-wise derivative of SiLU(g) * u, also restoring h
//   * pair_dot_kernel        the gradient of a combine weight: a dot product of two rows per pair
//   * router_backward_kernel combine-weight gradients -> logit gradients (sigmoid / softmax, with
//                            or without renormalisation over the selected experts)
// They are what torch.autograd derives from moe.py:102-157, experts.py:102-112 and ffn.py:374-395.
#include <type_traits>

#include "common.h"
#include "experts_f32.h"
#include "tile_map.h"

namespace fs2moe {

// ---------------------------------------------------------------------------------- weight gradient
// C_e [M, N] = sum over the rows r of expert e of A[r, :M]^T B[r, :N], bf16 (f32:
// grouped_wgrad_f32_kernel in experts_f32.h).  A block owns a 256 x 256 tile of one expert's gradient and
// walks the expert's rows 32 at a time.  Eight consumer waves multiply (a wave 128 x 64: 4 x 2 MFMA
// tiles); four producer waves, one per SIMD, move the data: a wave that waits for memory issues nothing
// else, so loads issued by the waves that multiply cost matrix-pipe time.  Both chunks go to LDS as they
// lie in memory (row = contraction index, columns contiguous) and come back through the transposing LDS
// read, in MFMA operand order.  LDS holds two chunks: while one is multiplied the producers write the
// next from registers and the two after that are on their way from memory in two sets of registers, so
// there is one barrier per chunk, which orders LDS traffic only.
// (Chunks of twice the rows, a half per register set and one barrier per chunk, were slower: 277
// against 244 us on 8 experts of 8192 rows.)  Rows past the expert's count are zero-filled,
// experts without rows get a zero gradient.
//
// Blocks are persistent, one per CU, and a launch may hold several gradients (WgradJobs).  Their tiles
// form one list: the gradients of one group (each slot a segment of its rows), then expert by expert all
// grouped gradients, inside a gradient bands of BAND row blocks of C, row block minor.  A tile costs its
// chunks and kTileCost more.  How the list is dealt depends on the largest tile:
//   * at most a quarter of a block's fair share: eight equal shares by cost, one per XCD; the blocks of the
//     XCD (block b runs on XCD b % 8) take the share's tiles in turn, so that at any time they work on
//     neighbours, which share operand slabs in the XCD's L2 (shares of neighbours per block instead: 2170
//     against 1750 us at 8 experts of 2048 rows, M 4096, N 14336);
//   * larger (a few experts or one group hold most rows): the tiles above that quarter go out one per block in rounds that
//     reverse direction, those of experts with the experts sorted by their rows, and the rest fill the blocks up to a
//     common level: each XCD gets a share as large as its blocks' room, and its blocks take the share's tiles in turn, each
//     from the round on that its large tiles last to.  As a share of neighbours for each block, a block for itself, every
//     tile read its operands from memory: 4096 tokens, top-8 of 128, 2048 x 768, evenly loaded with the router's gradient
//     2.37 GB for 2.42 that the tiles take in, now 0.55 (FETCH_SIZE 1.18 and 0.27, which counts requests of 128 bytes as
//     64), the launch under that counter 556 -> 523 us.  us of that training step with a norm 1581 -> 1549, by a popularity
//     law 1670 -> 1632; 8192 tokens 2526 -> 2444 and 2618 -> 2561.  Sorted only where experts have large tiles: in the gradients' order two operands share L2, not six.
// The chunks of a block's tiles form one stream: while the consumers write a tile out, the producers have
// the next one's first three chunks on their way.  (A block per tile, started by the hardware, paid about
// 10 us around its chunks.)
namespace wgk {
constexpr int TM = 256, TN = 256, CONSUMERS = 8, PRODUCERS = 4, WAVES = CONSUMERS + PRODUCERS;
constexpr int RK = 32;                                  // rows per chunk
constexpr int ROWB = TM * 2;                            // bytes per LDS row
constexpr int OPB = RK * ROWB;                          // bytes per operand chunk (16 KB)
constexpr int RING_BYTES = 4 * OPB;                     // two chunks of both operands
constexpr int LDE = 136;                                // epilogue: bytes between rows
constexpr int EPI_BYTES = CONSUMERS * 32 * LDE;         // a 32 x 64 piece per consumer
constexpr int MAX_BLOCKS = 512;
constexpr int TABLE_INTS = 4 * FS2MOE_MAX_EXPERTS + 4 + MAX_BLOCKS;
constexpr int SMEM_BYTES = RING_BYTES + EPI_BYTES + TABLE_INTS * 4;
// What a tile costs besides its chunks, in chunks: starting its accumulators and writing 128 KB.
constexpr int kTileCost = 5;
constexpr int BAND = 8;
constexpr int MAX_JOBS = 8;
}  // namespace wgk
// what a load through a row map reads past the end (not const: a global address, so the loads stay global
// loads)
static __device__ __attribute__((aligned(16))) uint32_t kZero16[4] = {0u, 0u, 0u, 0u};

// One gradient: slots of rows, one per expert (grouped), or segments of seg_rows rows of one group, whose
// f32 sums go to `partial` [slots, M, N] when it is not null.
struct WgradJob {
  const uint16_t *A, *B;
  uint16_t* C;
  float* partial;
  int M, N, m_tiles, tiles;  // tiles: per slot
  int grouped, slots, seg_rows, rows;
  int past_cache;  // store C past the caches (see nt_stores)
  int map_a, map_b;  // MAPPED: this operand's rows are read through the row map
};
struct WgradJobs {
  WgradJob job[wgk::MAX_JOBS];
  int n;
};

// MAPPED: operands of some gradients are read through the row map (rows of the layer's input, or of its
// output gradient, that no one has copied into expert order).  The map's entries are asked for two chunks ahead, by one
// load per wave right behind those of the chunk before the last, with which they arrive: nothing waits for them alone.
// (As scalar loads a chunk ahead every barrier waited for them with the LDS traffic.)  That, and a way out of a tile
// without branches and waits around its stores, us of the gradients of a training step: 4096 tokens, top-8 of 128
// skewed, 2048 x 768 648 -> 617; top-6 of 64, 2048 x 1024 465 -> 449; 2000, top-4 of 60 skewed, 1024 x 1408 181 -> 173;
// 300 of the first 246 -> 236; 4096 evenly, top-8 of 128 554 -> 553 (where memory then bound them, see the deal above).
// The map holds at least one entry, and one for every row of a gradient in the same launch that does not use it.
template <bool MAPPED>
__global__ __launch_bounds__(wgk::WAVES * 64) void grouped_wgrad_kernel(
    const WgradJobs jobs, const int32_t* __restrict__ row_map, const int32_t* __restrict__ counts,
    const int32_t* __restrict__ offsets, int E) {
  using namespace wgk;
  constexpr int ROW_CHUNKS = TM / 8;              // 16-byte chunks per LDS row (32)
  constexpr int PLANES = PRODUCERS * 64;          // lanes that move data
  constexpr int PER_THREAD = RK * ROW_CHUNKS / PLANES;  // chunks per producer lane and operand (4)
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  int32_t* s_cnt = reinterpret_cast<int32_t*>(smem + RING_BYTES + EPI_BYTES);
  int32_t* s_off = s_cnt + FS2MOE_MAX_EXPERTS;
  int32_t* s_exp = s_off + FS2MOE_MAX_EXPERTS;    // expert of list position
  int32_t* s_pre = s_exp + FS2MOE_MAX_EXPERTS;    // [E + 1]: chunks + kTileCost of the positions before
  int32_t* s_cap = s_pre + FS2MOE_MAX_EXPERTS + 4;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  __shared__ int s_wave_tot[WAVES], s_wave_max[WAVES];
  // The experts' tables in the order of `pos` (position of expert tid), and the prefix sums of their costs.
  const int my_cnt = counts != nullptr && tid < E ? counts[tid] : 0;
  const int my_off = counts != nullptr && tid < E ? offsets[tid] : 0;
  auto tables = [&](int pos) {
    if (tid < E) {
      s_cnt[pos] = my_cnt;
      s_off[pos] = my_off;
      s_exp[pos] = tid;
    }
    __syncthreads();
    const int cost = tid < E ? (s_cnt[tid] + RK - 1) / RK + kTileCost : 0;
    int incl = cost, most = cost;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(incl, off, kWave);
      if (lane >= off) incl += v;
    }
    most = (int)wave_max_u32((uint32_t)most);
    if (lane == 63) {
      s_wave_tot[wave] = incl;
      s_wave_max[wave] = most;
    }
    __syncthreads();
    int base = 0;
    for (int w = 0; w < wave; ++w) base += s_wave_tot[w];
    if (tid < E) {
      s_pre[tid] = base + incl - cost;
      if (tid == E - 1) s_pre[E] = base + incl;
    }
    __syncthreads();
  };
  if (counts != nullptr) tables(tid);
  // (a 64-bit division is some 150 instructions, and nearly every cost fits 32 bits)
  auto divide = [](int64_t n, int64_t d) -> int64_t {
    if (((n | d) >> 31) == 0) return (uint32_t)n / (uint32_t)d;
    return n / d;
  };
  // ---- the list: `dense` tiles of the gradients of one group, then those of the experts: gradient by
  // gradient (expert by expert the rows of three gradients, rather than two operands of one, would compete
  // for L2: 958 against 880 us for the gradients of 128 experts of 512 rows, 2048 x 768), or `per` tiles
  // for each expert where the experts are taken in the order of their sizes
  // (all segments of a gradient but the last have seg_rows rows)
  auto seg_cost = [&](const WgradJob& j, int slot) {
    const int left = j.rows - slot * j.seg_rows;
    return ((left < j.seg_rows ? left : j.seg_rows) + RK - 1) / RK + kTileCost;
  };
  int dense = 0, per = 0, most = 0;
  int64_t dense_cost = 0;
  for (int i = 0; i < jobs.n; ++i) {
    const WgradJob& j = jobs.job[i];
    if (j.grouped) {
      per += j.tiles;
      continue;
    }
    const int c = seg_cost(j, 0);
    dense += j.slots * j.tiles;
    dense_cost += ((int64_t)(j.slots - 1) * c + seg_cost(j, j.slots - 1)) * j.tiles;
    most = c > most ? c : most;
  }
  if (per > 0)
    for (int w = 0; w < WAVES; ++w) most = s_wave_max[w] > most ? s_wave_max[w] : most;
  const int64_t total = dense_cost + (per > 0 ? (int64_t)s_pre[E] * per : 0);
  bool by_expert = false;
  // The number of tiles whose middle lies before cost x of the list: where a share from x on begins.
  auto tiles_before = [&](int64_t x) -> int {
    int tiles = 0, tiles_of = per, cost;
    if (x < dense_cost) {
      for (int i = 0;; ++i) {
        const WgradJob& j = jobs.job[i];
        if (j.grouped) continue;
        const int c = seg_cost(j, 0), last = seg_cost(j, j.slots - 1);
        const int64_t all = ((int64_t)(j.slots - 1) * c + last) * j.tiles;
        if (x >= all) {
          x -= all;
          tiles += j.slots * j.tiles;
          continue;
        }
        int slot = (int)divide(x, (int64_t)c * j.tiles);
        slot = slot < j.slots - 1 ? slot : j.slots - 1;
        x -= (int64_t)slot * c * j.tiles;
        tiles += slot * j.tiles;
        tiles_of = j.tiles;
        cost = slot < j.slots - 1 ? c : last;
        break;
      }
    } else {
      x -= dense_cost;
      tiles = dense;
      if (per == 0 || x >= (int64_t)s_pre[E] * per) return dense + E * per;
      if (!by_expert)
        for (int i = 0;; ++i) {
          const WgradJob& j = jobs.job[i];
          if (!j.grouped) continue;
          tiles_of = j.tiles;
          const int64_t all = (int64_t)s_pre[E] * tiles_of;
          if (x < all) break;
          x -= all;
          tiles += E * tiles_of;
        }
      const int col = (int)divide(x, tiles_of);  // s_pre[pos] * tiles_of <= x  <=>  s_pre[pos] <= col
      int pos = 0;
      for (int e0 = 0; e0 < E; e0 += 64) {
        const int e = e0 + lane;
        const unsigned long long m = __ballot(e < E && s_pre[e] <= col && col < s_pre[e + 1]);
        if (m) pos = e0 + (int)__builtin_ctzll(m);
      }
      pos = __builtin_amdgcn_readfirstlane(pos);
      x -= (int64_t)s_pre[pos] * tiles_of;
      tiles += pos * tiles_of;
      cost = s_pre[pos + 1] - s_pre[pos];
    }
    // tile t of these begins at t cost; its middle lies before x for 2 t + 1 < 2 x / cost
    const int64_t t = divide(2 * x + cost - 1, 2 * (int64_t)cost);
    return tiles + (int)(t < tiles_of ? t : tiles_of);
  };
  // The block's tiles: `rounds` of one of the first `big` tiles each, then its XCD's tiles [next_t, end) in turn with the
  // XCD's other blocks: in rounds of one tile each, of which block i misses the first skip_i.  Of the tiles that go out
  // before the block's round n those of lane i's block are max(0, n + ahead).
  struct Deal {
    int slot, grid, rounds, big, round, next_t, end, turn, ahead;
    __device__ int next() {  // -1: no more
      while (round < rounds) {
        const int r = round++, p = r * grid + ((r & 1) ? grid - 1 - slot : slot);
        if (p < big) return p;
      }
      const int of_lane = turn + ahead, t = next_t + wave_sum_i32(of_lane > 0 ? of_lane : 0);
      ++turn;
      return t < end ? t : -1;
    }
  };
  Deal deal;
  deal.grid = (int)gridDim.x;
  const int xcd = blockIdx.x & 7;
  deal.slot = xcd * (deal.grid >> 3) + (int)(blockIdx.x >> 3);
  deal.round = deal.rounds = deal.big = deal.turn = 0;
  // (nothing skipped: the blocks before this one are a tile ahead; lanes without a block never count)
  constexpr int NEVER = -(1 << 29);
  const int xcd_blocks = deal.grid >> 3, rank = (int)(blockIdx.x >> 3);
  deal.ahead = lane < xcd_blocks ? (lane < rank ? 1 : 0) : NEVER;
  const int64_t fair = divide(total, deal.grid);
  if (dense + (int64_t)E * per <= deal.grid) {
    deal.big = dense + E * per;  // at most one tile each
    deal.rounds = 1;
    deal.next_t = deal.end = 0;
  } else if (most * 4ll <= fair) {
    deal.next_t = tiles_before(total * xcd / 8);
    deal.end = tiles_before(total * (xcd + 1) / 8);
  } else {
    int expert_most = 0;
    for (int w = 0; per > 0 && w < WAVES; ++w) expert_most = s_wave_max[w] > expert_most ? s_wave_max[w] : expert_most;
    // (where only the gradients of one group have large tiles, the others stay in the order that shares operands best)
    by_expert = expert_most * 4ll > fair;
    if (by_expert) {
      // sort the experts by their rows, largest first (ties: lower index first)
      int rank = 0;
      for (int j = 0; j < E; ++j) {
        const int cj = s_cnt[j];
        rank += (cj > my_cnt || (cj == my_cnt && j < tid)) ? 1 : 0;
      }
      __syncthreads();
      tables(rank);
    }
    // the large tiles: all of one group (as large as any expert's, mostly), and the experts whose tiles
    // are above a quarter of the fair share
    int large = 0;
    if (by_expert) {
      for (int e0 = 0; e0 < E; e0 += 64) {
        const int e = e0 + lane;
        large += __popcll(__ballot(e < E && (s_pre[e + 1] - s_pre[e]) * 4ll > fair));
      }
    }
    deal.big = dense + large * per;
    deal.rounds = (deal.big + deal.grid - 1) / deal.grid;
    const int64_t big_cost = dense_cost + (large > 0 ? (int64_t)s_pre[large] * per : 0);
    // the load of every block (by slot) after the rounds
    for (int sl = tid; sl < deal.grid; sl += WAVES * 64) {
      int load = 0;
      for (int r = 0; r < deal.rounds; ++r) {
        const int p = r * deal.grid + ((r & 1) ? deal.grid - 1 - sl : sl);
        if (p >= deal.big) continue;
        if (p >= dense) {
          const int pos = (p - dense) / per;
          load += s_pre[pos + 1] - s_pre[pos];
        } else {
          int q = p, i = 0;
          for (;; ++i) {
            const WgradJob& j = jobs.job[i];
            if (j.grouped) continue;
            if (q < j.slots * j.tiles) {
              load += seg_cost(j, q / j.tiles);
              break;
            }
            q -= j.slots * j.tiles;
          }
        }
      }
      s_cap[sl] = load;
    }
    __syncthreads();
    // The level L that the remaining cost fills the blocks to, L = (rest + loads below L) / (blocks below
    // L): from all blocks on, dropping those above, until none is; then this block's part of what lies
    // between the loads and L.  Every wave for itself, lane l holding the loads of slots 8 l .. 8 l + 7.
    const int64_t rest = total - big_cost;
    constexpr int PL = MAX_BLOCKS / 64;
    int load[PL];
#pragma unroll
    for (int i = 0; i < PL; ++i) load[i] = PL * lane + i < deal.grid ? s_cap[PL * lane + i] : 0x7fffffff;
    int level = 0x7ffffffe;
    for (int below = deal.grid + 1;;) {
      int n = 0, sum = 0;
#pragma unroll
      for (int i = 0; i < PL; ++i)
        if (load[i] <= level) {
          ++n;
          sum += load[i];
        }
      n = wave_sum_i32(n);
      if (n == below) break;
      below = n;
      level = (int)divide(rest + wave_sum_i32(sum) + n - 1, n);
    }
    // the XCD's part of it: the room of its blocks behind that of the XCDs before
    const int first_slot = xcd * xcd_blocks;
    int mine = 0, before = 0;
#pragma unroll
    for (int i = 0; i < PL; ++i) {
      const int r = load[i] <= level ? level - load[i] : 0, sl = PL * lane + i;
      if (sl < first_slot) before += r;
      if (sl >= first_slot && sl < first_slot + xcd_blocks) mine += r;
    }
    const int64_t from = wave_sum_i32(before), room = wave_sum_i32(mine), to = from + room;
    const int64_t first_cost = big_cost + (from < rest ? from : rest);
    deal.next_t = tiles_before(first_cost);
    deal.end = tiles_before(big_cost + (to < rest ? to : rest));
    // A block joins the XCD's rounds when the others have been filled to its load: as many rounds as tiles of that cost
    // lie at the share's beginning, for the number of blocks that take part on average.
    const int my_load = lane < xcd_blocks ? s_cap[first_slot + lane] : 0x7fffffff;
    const int least = -(int)wave_max_u32((uint32_t)(0x7fffffff - my_load)) + 0x7fffffff, height = level - least;
    const int part = height > 0 ? (int)divide(room + height - 1, height) : 0;  // blocks
    int skip = 0;
    if (my_load >= level) {
      skip = -NEVER;
    } else if (per > 0 && my_load > least) {
      int64_t y = first_cost - dense_cost + (int64_t)part * (my_load - least);
      int tiles = dense, tiles_of = per;
      if (!by_expert)
        for (int i = 0; i < jobs.n; ++i) {
          const WgradJob& j = jobs.job[i];
          if (!j.grouped) continue;
          tiles_of = j.tiles;
          const int64_t all = (int64_t)s_pre[E] * tiles_of;
          if (y < all) break;
          y -= all;
          tiles += E * tiles_of;
        }
      int lo = 0, hi = E;  // the expert of cost y
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if ((int64_t)s_pre[mid] * tiles_of <= y) lo = mid;
        else hi = mid;
      }
      const int64_t in = y - (int64_t)s_pre[lo] * tiles_of;
      tiles += lo * tiles_of + (int)divide(in, s_pre[lo + 1] - s_pre[lo]) - deal.next_t;
      skip = tiles > 0 ? (2 * tiles + part) / (2 * part) : 0;
    }
    if (lane < xcd_blocks) {
      const int own = __builtin_amdgcn_readlane(skip, rank);
      deal.ahead = skip == -NEVER || own == -NEVER ? NEVER : own - skip + (lane < rank ? 1 : 0);
      if (own == -NEVER) deal.end = deal.next_t;
    }
    deal.end = __builtin_amdgcn_readfirstlane(deal.end);
  }
  deal.next_t = __builtin_amdgcn_readfirstlane(deal.next_t);
  deal.end = __builtin_amdgcn_readfirstlane(deal.end);
  // (all of it is the same in every lane, but was computed from LDS: as scalars from here on, or the loops
  // over tiles and chunks would be masked ones, whose paths meet where nothing can be known of the loads)
  deal.rounds = __builtin_amdgcn_readfirstlane(deal.rounds);
  deal.big = __builtin_amdgcn_readfirstlane(deal.big);
  by_expert = __builtin_amdgcn_readfirstlane(by_expert);

  auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  // Wave-uniform parameters of a tile.
  struct Tile {
    int job, slot, off, cnt, m0, n0;
  };
  auto locate = [&](int t) {
    Tile r;
    int pos = 0;
    const bool grouped = t >= dense;
    if (grouped) {
      t -= dense;
      if (by_expert) {
        pos = t / per;
        t -= pos * per;
      }
    }
    for (r.job = 0;; ++r.job) {
      const WgradJob& j = jobs.job[r.job];
      if ((j.grouped != 0) != grouped) continue;
      const int n = grouped && by_expert ? j.tiles : j.slots * j.tiles;
      if (t < n) break;
      t -= n;
    }
    const WgradJob& j = jobs.job[r.job];
    if (grouped && !by_expert) {
      pos = t / j.tiles;
      t -= pos * j.tiles;
    }
    if (grouped) {
      r.slot = __builtin_amdgcn_readfirstlane(s_exp[pos]);
      r.off = __builtin_amdgcn_readfirstlane(s_off[pos]);
      r.cnt = __builtin_amdgcn_readfirstlane(s_cnt[pos]);
    } else {
      r.slot = t / j.tiles;
      t -= r.slot * j.tiles;
      r.off = r.slot * j.seg_rows;
      r.cnt = j.rows - r.off < j.seg_rows ? j.rows - r.off : j.seg_rows;
    }
    const int n_tiles = j.tiles / j.m_tiles, band = t / (BAND * n_tiles);
    const int i = t - band * BAND * n_tiles, left = j.m_tiles - band * BAND;
    const int high = left < BAND ? left : BAND, nt = i / high;
    r.m0 = (band * BAND + i - nt * high) * TM;
    r.n0 = nt * TN;
    return r;
  };

  if (wave >= CONSUMERS) {
    // ---- producers: chunk g of the block's stream goes to LDS buffer g & 1 through register set g & 1;
    // while chunk g is multiplied, chunk g + 1 goes into the other buffer (read last during chunk g - 1:
    // the barrier that ended it has passed), chunk g + 3 is loaded into the set this frees, and chunk
    // g + 2 is still on its way in the other set.  Every load and store is unconditional (what lies past
    // a tile's rows or columns, or past the stream's end, loads zeros: an offset outside the buffer):
    // behind a condition the compiler cannot count the loads in flight, and waits for all of them, the
    // other set's included, before a store.
    const int ptid = tid - CONSUMERS * 64;
    const int kr = ptid / ROW_CHUNKS, ch = ptid % ROW_CHUNKS;  // rows kr + 8 i, chunk ch
    u32x4 ra[2][PER_THREAD], rb[2][PER_THREAD];
    // the chunk to load next: rows [ld_off, ld_off + ld_left) of the tile's operands
    const uint16_t* ld_a = nullptr;
    const uint16_t* ld_b = nullptr;
    int ld_left = 0, ld_lda = 0, ld_ldb = 0;
    // MAPPED: the chunk's first row in expert order, which operands go through the map, a lane's place in row 0 of the
    // operands, and their rows' distance
    typedef u32x4 __attribute__((address_space(1))) GlobalVec;
    uint64_t zero = (uint64_t)kZero16;
    asm volatile("" : "+s"(zero));  // (read once)
    int ld_row = 0, ld_map_a = 0, ld_map_b = 0;
    uint64_t row_a = zero, row_b = zero;
    uint32_t pitch_a = 0, pitch_b = 0;
    // and the same of the next chunk to load into each register set, with its rows' entries: lane l holds row kr + 8 (l & 3)'s
    struct Ahead {
      uint64_t row_a, row_b;
      uint32_t pitch_a, pitch_b;
      int row, left, map_a, map_b, entry;
    } next_up[2];
    Deal ld_deal = deal;
    uint32_t oa[PER_THREAD], ob[PER_THREAD];
    int loaded = 0;  // chunks so far (those past the stream's end do not count)
    auto next_tile = [&]() {
      // (tiles without rows have no chunks)
      ld_left = 0;
      for (int n; ld_left == 0 && (n = uniform(ld_deal.next())) >= 0;) {
        const Tile t = locate(n);
        if (t.cnt == 0) continue;
        const WgradJob& j = jobs.job[t.job];
        ld_lda = j.M;
        ld_ldb = j.N;
        ld_a = (MAPPED ? j.A : j.A + (size_t)t.off * j.M) + t.m0;
        ld_b = (MAPPED ? j.B : j.B + (size_t)t.off * j.N) + t.n0;
        ld_row = t.off;
        ld_map_a = j.map_a;
        ld_map_b = j.map_b;
        ld_left = t.cnt;
        // (columns past the operand's: all ones, past any buffer's end.  As selects these become branches,
        // at whose joins the tile's parameters stop being scalars)
        uint32_t a_out = t.m0 + ch * 8 < j.M ? 0u : 0xfffffff0u, b_out = t.n0 + ch * 8 < j.N ? 0u : 0xfffffff0u;
        asm volatile("" : "+v"(a_out), "+v"(b_out));
        if constexpr (MAPPED) {
          row_a = a_out == 0u ? (uint64_t)ld_a + ch * 16 : zero;
          row_b = b_out == 0u ? (uint64_t)ld_b + ch * 16 : zero;
          pitch_a = a_out == 0u ? (uint32_t)j.M * 2u : 0u;
          pitch_b = b_out == 0u ? (uint32_t)j.N * 2u : 0u;
          continue;
        }
#pragma unroll
        for (int i = 0; i < PER_THREAD; ++i) {
          oa[i] = (uint32_t)(((kr + 8 * i) * j.M + ch * 8) * 2) | a_out;
          ob[i] = (uint32_t)(((kr + 8 * i) * j.N + ch * 8) * 2) | b_out;
        }
      }
    };
    auto scalar = [&](const uint16_t* q) {
      const uint64_t v = (uint64_t)q;
      return (uint16_t*)((uint64_t)(uint32_t)uniform((int)(v >> 32)) << 32 | (uint32_t)uniform((int)v));
    };
    // MAPPED: the stream's next chunk becomes the register set's, and its entries are asked for.
    auto look_up = [&](auto set_c) {
      if constexpr (MAPPED) {
        if (uniform(ld_left) <= 0) next_tile();
        const int k = kr + 8 * (lane & 3), last = ld_left - 1;
        const int entry = row_map[last >= 0 ? ld_row + (k < last ? k : last) : 0];
        next_up[decltype(set_c)::value] = {row_a, row_b, pitch_a, pitch_b, ld_row, ld_left, ld_map_a, ld_map_b, entry};
        loaded += (int)((uint32_t)-ld_left >> 31);  // (as below)
        ld_row += RK;
        ld_left -= RK;
      }
    };
    // MAPPED: where the chunk's pieces lie.
    // (a lane whose column lies past the operand's reads zeros whatever the row)
    uint64_t at_a[PER_THREAD], at_b[PER_THREAD];
    auto place_chunk = [&](auto set_c) {
      if constexpr (MAPPED) {
        const Ahead& up = next_up[decltype(set_c)::value];
        const int left = uniform(up.left), last = left - 1;
#pragma unroll
        for (int i = 0; i < PER_THREAD; ++i) {
          const uint32_t e0 = __builtin_amdgcn_readlane(up.entry, i), e1 = __builtin_amdgcn_readlane(up.entry, 32 + i);
          const int k = kr + 8 * i;
          const uint32_t mapped = lane < 32 ? e0 : e1, place = last >= 0 ? up.row + (k < last ? k : last) : 0;
          at_a[i] = up.row_a + (uint64_t)(up.map_a ? mapped : place) * up.pitch_a;
          at_b[i] = up.row_b + (uint64_t)(up.map_b ? mapped : place) * up.pitch_b;
        }
        if (left < RK) {
#pragma unroll
          for (int i = 0; i < PER_THREAD; ++i) {
            const bool in = kr + 8 * i < left;
            at_a[i] = in ? at_a[i] : zero;
            at_b[i] = in ? at_b[i] : zero;
          }
        }
#pragma unroll
        for (int i = 0; i < PER_THREAD; ++i) asm volatile("" : "+v"(at_a[i]), "+v"(at_b[i]));
      }
    };
    auto load_chunk = [&](auto set_c) {
      constexpr int set = decltype(set_c)::value;
      if constexpr (MAPPED) {
#pragma unroll
        for (int i = 0; i < PER_THREAD; ++i) {
          ra[set][i] = *(const GlobalVec*)at_a[i];
          rb[set][i] = *(const GlobalVec*)at_b[i];
        }
      } else {
        // one more if ld_left > 0 (a truth value is added on the vector side, and takes the loop's end with it)
        loaded += (int)((uint32_t)-ld_left >> 31);
        const __amdgpu_buffer_rsrc_t a_rsrc =
            __builtin_amdgcn_make_buffer_rsrc(scalar(ld_a), 0, 0xfffffff0u, 0x00020000);
        const __amdgpu_buffer_rsrc_t b_rsrc =
            __builtin_amdgcn_make_buffer_rsrc(scalar(ld_b), 0, 0xfffffff0u, 0x00020000);
#pragma unroll
        for (int i = 0; i < PER_THREAD; ++i) {
          const bool in = kr + 8 * i < ld_left;
          uint32_t at_a = in ? oa[i] : 0xfffffff0u, at_b = in ? ob[i] : 0xfffffff0u;
          asm volatile("" : "+v"(at_a), "+v"(at_b));  // (chosen before the load, not by branches around two)
          ra[set][i] = __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, at_a, 0, 0);
          rb[set][i] = __builtin_amdgcn_raw_buffer_load_b128(b_rsrc, at_b, 0, 0);
        }
        ld_a += (size_t)RK * ld_lda;
        ld_b += (size_t)RK * ld_ldb;
        ld_left -= RK;
        if (uniform(ld_left) <= 0) next_tile();
      }
    };
    auto store_chunk = [&](auto set_c, int buf) {
      constexpr int set = decltype(set_c)::value;
      uint8_t* sA = smem + buf * 2 * OPB;
      uint8_t* sB = sA + OPB;
#pragma unroll
      for (int i = 0; i < PER_THREAD; ++i) {
        // chunk ch of row k sits in slot ch ^ ((k & 3) << 2), so that the four consecutive rows a
        // transposing read touches lie 64 bytes apart
        const int k = kr + 8 * i, at = k * ROWB + ((ch ^ ((k & 3) << 2)) * 16);
        *reinterpret_cast<u32x4*>(sA + at) = ra[set][i];
        *reinterpret_cast<u32x4*>(sB + at) = rb[set][i];
      }
    };
    using Set0 = std::integral_constant<int, 0>;
    using Set1 = std::integral_constant<int, 1>;
    if constexpr (MAPPED) {
      look_up(Set0{});
      look_up(Set1{});
    } else {
      next_tile();
    }
    place_chunk(Set0{});
    load_chunk(Set0{});
    if (loaded == 0) return;  // no tile with rows: nothing for the consumers to wait for
    look_up(Set0{});
    place_chunk(Set1{});
    load_chunk(Set1{});
    look_up(Set1{});
    store_chunk(Set0{}, 0);
    place_chunk(Set0{});
    load_chunk(Set0{});
    look_up(Set0{});
    lds_barrier();
    auto step = [&](int g, auto next_set) {
      store_chunk(next_set, (g + 1) & 1);
      place_chunk(next_set);
      load_chunk(next_set);
      look_up(next_set);
      lds_barrier();  // the loads of the next chunks stay in flight
    };
    // Always two steps, the one past an odd last chunk with zeros that no one reads, and everything that the
    // loop's way depends on in scalars: where a skipped step's path, or a masked lane's, joined the loop again
    // the compiler waited for all loads in flight, in every other step.  128 experts of about 256 rows, 2048 x
    // 768, 189 -> 178 us; 8 of 2048, 4096 x 14336, 1775 -> 1655; 60 of 300, 1096 x 1416, 116 -> 106.  (A
    // third set of registers gives the long ones nothing more and costs launches of few chunks 1 to 2 us.)
    for (int g = 0; g < uniform(loaded); g += 2) {  // (a step's load is three chunks ahead: `loaded` is final)
      step(g, Set1{});
      step(g + 1, Set0{});
    }
    return;  // the consumers write the tiles
  }

  // ---- consumers
  const int wm = wave & 1, wn = (wave >> 1) & 3;  // a consumer's 128 (m) x 64 (n) part of the tile
  const int lr = lane & 31, lk = lane >> 5;
  // fragment address of the 32 columns from cbase on, rows 8 lk .. 8 lk + 3 (+4 for the upper half)
  auto tr_addr = [&](int cbase) {
    const int s = lane & 15, half = (lane >> 4) & 1;
    const int k = lk * 8 + (s >> 2);
    const int col = cbase + half * 16 + (s & 3) * 4;
    return k * ROWB + (((col >> 3) ^ ((k & 3) << 2)) * 16) + (col & 7) * 2;
  };
  int fa[4], fb[2];
#pragma unroll
  for (int t = 0; t < 4; ++t) fa[t] = tr_addr(wm * 128 + t * 32);
#pragma unroll
  for (int t = 0; t < 2; ++t) fb[t] = tr_addr(wn * 64 + t * 32);

  f32x16 acc[2][4];  // [tn][tm]
  auto compute_chunk = [&](int buf) {
    const uint8_t* sA = smem + buf * 2 * OPB;
    const uint8_t* sB = sA + OPB;
#pragma unroll
    for (int ks = 0; ks < RK / 16; ++ks) {
      bf16x8 af[4], bfr[2];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const uint8_t* pa = sA + fa[t] + ks * 16 * ROWB;
        af[t] = lds_read_frag_tr(reinterpret_cast<const uint16_t*>(pa),
                                 reinterpret_cast<const uint16_t*>(pa + 4 * ROWB));
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const uint8_t* pb = sB + fb[t] + ks * 16 * ROWB;
        bfr[t] = lds_read_frag_tr(reinterpret_cast<const uint16_t*>(pb),
                                  reinterpret_cast<const uint16_t*>(pb + 4 * ROWB));
      }
#pragma unroll
      for (int tn = 0; tn < 2; ++tn)
#pragma unroll
        for (int tm = 0; tm < 4; ++tm)
          acc[tn][tm] =
              __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[tn], af[tm], acc[tn][tm], 0, 0, 0);
    }
  };
  // Accumulator layout: the lane holds row m = lr of fragment tm and columns 8 q + 4 lk + {0..3} of
  // fragment tn in registers 4 q .. 4 q + 3.
  auto write_tile = [&](const Tile& tl) {
    const WgradJob& j = jobs.job[tl.job];
    const int M = j.M, N = j.N;
    if (j.partial == nullptr) {
      // Through the wave's own piece of LDS, so that a store instruction writes 8 rows of 128 contiguous
      // bytes instead of 32 rows of 16: a 32 (m) x 64 (n) fragment row as bf16, rows 136 bytes apart,
      // read back 16 bytes per lane.
      // (rows past the matrix lie past the buffer's end, and lanes whose columns do stay at an offset there: N is a
      // multiple of 8, so the eight columns are in or out together.  The host keeps every offset of a tile's rows below)
      const int rows = M - tl.m0 < TM ? M - tl.m0 : TM;
      const __amdgpu_buffer_rsrc_t c_rsrc =
          __builtin_amdgcn_make_buffer_rsrc(j.C + (size_t)tl.slot * M * N + (size_t)tl.m0 * N + tl.n0, 0,
                                            (int)(((uint32_t)rows * N - tl.n0) * 2u), 0x00020000);
      uint8_t* sw = smem + RING_BYTES + wave * 32 * LDE;
      const int rrow = lane >> 3, rcol = lane & 7, col = wn * 64 + rcol * 8;
      const bool in = tl.n0 + col < N;
      const uint32_t at = in ? ((uint32_t)(wm * 128 + rrow) * N + col) * 2u : 0xfffffff0u, rows8 = in ? N * 16u : 0u;
      auto write = [&](auto past) {
#pragma unroll
        for (int tm = 0; tm < 4; ++tm) {
#pragma unroll
          for (int tn = 0; tn < 2; ++tn)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              u32x2 o = {pack_bf16x2(acc[tn][tm][4 * q], acc[tn][tm][4 * q + 1]),
                         pack_bf16x2(acc[tn][tm][4 * q + 2], acc[tn][tm][4 * q + 3])};
              *reinterpret_cast<u32x2*>(sw + lr * LDE + (tn * 32 + 8 * q + 4 * lk) * 2) = o;
            }
          // the wave's own LDS traffic runs in order; the compiler must not move the reads (other
          // lanes' data) above the writes, nor the next round's writes above these reads
          asm volatile("" ::: "memory");
          u32x4 o[4];
#pragma unroll
          for (int p8 = 0; p8 < 4; ++p8) {
            const uint8_t* from = sw + (p8 * 8 + rrow) * LDE + rcol * 16;
            const u32x2 lo = *reinterpret_cast<const u32x2*>(from), hi = *reinterpret_cast<const u32x2*>(from + 8);
            o[p8] = u32x4{lo[0], lo[1], hi[0], hi[1]};
          }
          asm volatile("" ::: "memory");
#pragma unroll
          for (int p8 = 0; p8 < 4; ++p8)
            __builtin_amdgcn_raw_buffer_store_b128(o[p8], c_rsrc, (int)(at + (uint32_t)(tm * 4 + p8) * rows8), 0,
                                                   decltype(past)::value ? kNonTemporal : 0);
        }
      };
      if (j.past_cache)
        write(std::true_type{});
      else
        write(std::false_type{});
      return;
    }
    float* Pe = j.partial + (size_t)tl.slot * M * N;
#pragma unroll
    for (int tm = 0; tm < 4; ++tm) {
      const int m = tl.m0 + wm * 128 + tm * 32 + lr;
      if (m >= M) continue;
#pragma unroll
      for (int tn = 0; tn < 2; ++tn) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = tl.n0 + wn * 64 + tn * 32 + 8 * q + 4 * lk;
          if (n >= N) continue;  // N is a multiple of 4: the four columns are in or out together
          f32x4 o = {acc[tn][tm][4 * q], acc[tn][tm][4 * q + 1], acc[tn][tm][4 * q + 2],
                     acc[tn][tm][4 * q + 3]};
          *reinterpret_cast<f32x4*>(Pe + (size_t)m * N + n) = o;
        }
      }
    }
  };
  bool started = false;
  int buf = 0, chunks_done = 0;
  for (int n; (n = deal.next()) >= 0;) {
    const Tile tl = locate(n);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;
    const int chunks = (tl.cnt + RK - 1) / RK;
    if (chunks > 0 && !started) {
      lds_barrier();
      started = true;
    }
    for (int i = 0; i < chunks; ++i) {
      compute_chunk(buf);
      buf ^= 1;
      ++chunks_done;
      lds_barrier();
    }
    write_tile(tl);
  }
  if (chunks_done % 2 != 0) lds_barrier();  // the producers' last step
}

// out[i] = sum over the segments, in order, of partial[s][i]; one rounding.
template <typename T>
__global__ __launch_bounds__(256) void wgrad_reduce_kernel(const float* __restrict__ partial,
                                                           int segments, int64_t n,
                                                           T* __restrict__ out) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;  // n is a multiple of 4
  f32x4 acc = *reinterpret_cast<const f32x4*>(partial + i);
  for (int s = 1; s < segments; ++s) acc += *reinterpret_cast<const f32x4*>(partial + (size_t)s * n + i);
  if constexpr (sizeof(T) == 2) {
    u32x2 o = {pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3])};
    *reinterpret_cast<u32x2*>(out + i) = o;
  } else {
    *reinterpret_cast<f32x4*>(out + i) = acc;
  }
}

// ------------------------------------------------------------------------- SwiGLU, element-wise
// h = SiLU(g) * u;  dg = dh * u * s * (1 + g * (1 - s)),  du = dh * SiLU(g),  s = sigmoid(g).
// In f32 with one rounding per output; outputs may alias the inputs element for element.
template <typename T>
__global__ __launch_bounds__(256) void swiglu_backward_kernel(const T* g, const T* u, const T* dh,
                                                              int64_t n, T* h, T* dg, T* du) {
  constexpr int VEC = 16 / sizeof(T);
  const int64_t stride = (int64_t)gridDim.x * blockDim.x * VEC;
  for (int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * VEC; i < n; i += stride) {
    const u32x4 gv = *reinterpret_cast<const u32x4*>(g + i);
    const u32x4 uv = *reinterpret_cast<const u32x4*>(u + i);
    const u32x4 dv = *reinterpret_cast<const u32x4*>(dh + i);
    float gf[VEC], uf[VEC], df[VEC], ho[VEC], go[VEC], uo[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      if constexpr (sizeof(T) == 2) {
        const uint32_t gw = gv[j >> 1], uw = uv[j >> 1], dw = dv[j >> 1];
        gf[j] = __uint_as_float((j & 1) ? (gw & 0xffff0000u) : (gw << 16));
        uf[j] = __uint_as_float((j & 1) ? (uw & 0xffff0000u) : (uw << 16));
        df[j] = __uint_as_float((j & 1) ? (dw & 0xffff0000u) : (dw << 16));
      } else {
        gf[j] = __uint_as_float(gv[j]);
        uf[j] = __uint_as_float(uv[j]);
        df[j] = __uint_as_float(dv[j]);
      }
      const float s = 1.0f / (1.0f + __expf(-gf[j]));
      const float silu = gf[j] * s;
      ho[j] = silu * uf[j];
      go[j] = df[j] * uf[j] * (s * (1.0f + gf[j] * (1.0f - s)));
      uo[j] = df[j] * silu;
    }
    u32x4 hv, gov, uov;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (sizeof(T) == 2) {
        hv[j] = pack_bf16x2(ho[2 * j], ho[2 * j + 1]);
        gov[j] = pack_bf16x2(go[2 * j], go[2 * j + 1]);
        uov[j] = pack_bf16x2(uo[2 * j], uo[2 * j + 1]);
      } else {
        hv[j] = __float_as_uint(ho[j]);
        gov[j] = __float_as_uint(go[j]);
        uov[j] = __float_as_uint(uo[j]);
      }
    }
    *reinterpret_cast<u32x4*>(h + i) = hv;
    *reinterpret_cast<u32x4*>(dg + i) = gov;
    *reinterpret_cast<u32x4*>(du + i) = uov;
  }
}

// ------------------------------------------------------------------- gradient of a combine weight
// out[p] = <a[a_rows[p]], b[p / K]> (+ <a2[a_rows[p]], b[p / K]>) for the T*K pairs p: one wave per
// pair, f32 accumulation in a fixed order.
template <typename T>
__global__ __launch_bounds__(256) void pair_dot_kernel(const T* __restrict__ a,
                                                       const T* __restrict__ a2,
                                                       const int32_t* __restrict__ a_rows,
                                                       const T* __restrict__ b, int pairs, int K,
                                                       int D, int vec_ok, float* __restrict__ out) {
  const int p = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (p >= pairs) return;
  const int lane = threadIdx.x & 63;
  // A pair whose expert id was out of range has no row (dispatch wrote -1 for it, and combine
  // skips it): its weight contributed nothing, so its gradient is zero.  Uniform over the wave.
  const int row = a_rows[p];
  if (row < 0) {
    if (lane == 0) out[p] = 0.f;
    return;
  }
  const size_t ar = (size_t)row * D, br = (size_t)(p / K) * D;
  float s = 0.f;
  constexpr int VEC = 16 / sizeof(T);
  if (vec_ok) {
    // 16 bytes per lane and load
    for (int d = lane * VEC; d < D; d += 64 * VEC) {
      const u32x4 av = *reinterpret_cast<const u32x4*>(a + ar + d);
      const u32x4 bv = *reinterpret_cast<const u32x4*>(b + br + d);
      u32x4 cv = {0u, 0u, 0u, 0u};
      if (a2 != nullptr) cv = *reinterpret_cast<const u32x4*>(a2 + ar + d);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (sizeof(T) == 2) {
          float x0 = __uint_as_float(av[j] << 16), x1 = __uint_as_float(av[j] & 0xffff0000u);
          if (a2 != nullptr) {
            x0 += __uint_as_float(cv[j] << 16);
            x1 += __uint_as_float(cv[j] & 0xffff0000u);
          }
          s += x0 * __uint_as_float(bv[j] << 16);
          s += x1 * __uint_as_float(bv[j] & 0xffff0000u);
        } else {
          float x0 = __uint_as_float(av[j]);
          if (a2 != nullptr) x0 += __uint_as_float(cv[j]);
          s += x0 * __uint_as_float(bv[j]);
        }
      }
    }
  } else {
    for (int d = lane; d < D; d += 64) {
      float av = Elem<T>::load(a + ar + d);
      if (a2 != nullptr) av += Elem<T>::load(a2 + ar + d);
      s += av * Elem<T>::load(b + br + d);
    }
  }
  s = wave_sum_f32(s);
  if (lane == 0) out[p] = s;
}

// ------------------------------------------------------------------- RMS normalisation backward
// y = x r w with r = rsqrt(mean(x^2) + eps) (nn/normalization.py:234-236).  With gy = dy w:
//   dx = r gy - x r^3 <gy, x> / D        dw[j] = sum_t dy[t, j] x[t, j] r_t
// One wave per row, two passes over it (the second finds the row in cache); everything in f32,
// one rounding per stored element.  The row's r goes to rstd (may be null) for the weight gradient.
template <typename T>
__global__ __launch_bounds__(256) void rms_norm_backward_rows_kernel(
    const T* __restrict__ x, const T* __restrict__ w, float eps, const T* __restrict__ dy, int rows,
    int D, T* __restrict__ dx, float* __restrict__ rstd) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  constexpr int VEC = 16 / sizeof(T);
  const bool vec = D % VEC == 0;  // the host checks the alignment of the bases
  const float inv_d = 1.0f / (float)D;
  for (int t = blockIdx.x * 4 + wave; t < rows; t += gridDim.x * 4) {
    const T* xr = x + (size_t)t * D;
    const T* gr = dy + (size_t)t * D;
    T* outr = dx + (size_t)t * D;
    float ss = 0.f, sg = 0.f;
    if (vec) {
      for (int d = lane * VEC; d < D; d += 64 * VEC) {
        const u32x4 xv = *reinterpret_cast<const u32x4*>(xr + d);
        const u32x4 gv = *reinterpret_cast<const u32x4*>(gr + d);
        u32x4 wv = {0u, 0u, 0u, 0u};
        if (w != nullptr) wv = *reinterpret_cast<const u32x4*>(w + d);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (sizeof(T) == 2) {
            const float x0 = __uint_as_float(xv[j] << 16), x1 = __uint_as_float(xv[j] & 0xffff0000u);
            float g0 = __uint_as_float(gv[j] << 16), g1 = __uint_as_float(gv[j] & 0xffff0000u);
            if (w != nullptr) {
              g0 *= __uint_as_float(wv[j] << 16);
              g1 *= __uint_as_float(wv[j] & 0xffff0000u);
            }
            ss += x0 * x0;
            ss += x1 * x1;
            sg += g0 * x0;
            sg += g1 * x1;
          } else {
            const float x0 = __uint_as_float(xv[j]);
            float g0 = __uint_as_float(gv[j]);
            if (w != nullptr) g0 *= __uint_as_float(wv[j]);
            ss += x0 * x0;
            sg += g0 * x0;
          }
        }
      }
    } else {
      for (int d = lane; d < D; d += 64) {
        const float x0 = Elem<T>::load(xr + d);
        float g0 = Elem<T>::load(gr + d);
        if (w != nullptr) g0 *= Elem<T>::load(w + d);
        ss += x0 * x0;
        sg += g0 * x0;
      }
    }
    const float r = 1.0f / sqrtf(wave_sum_f32(ss) * inv_d + eps);
    const float c = r * r * r * wave_sum_f32(sg) * inv_d;
    if (rstd != nullptr && lane == 0) rstd[t] = r;
    if (vec) {
      for (int d = lane * VEC; d < D; d += 64 * VEC) {
        const u32x4 xv = *reinterpret_cast<const u32x4*>(xr + d);
        const u32x4 gv = *reinterpret_cast<const u32x4*>(gr + d);
        u32x4 wv = {0u, 0u, 0u, 0u};
        if (w != nullptr) wv = *reinterpret_cast<const u32x4*>(w + d);
        u32x4 ov;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (sizeof(T) == 2) {
            const float x0 = __uint_as_float(xv[j] << 16), x1 = __uint_as_float(xv[j] & 0xffff0000u);
            float g0 = __uint_as_float(gv[j] << 16), g1 = __uint_as_float(gv[j] & 0xffff0000u);
            if (w != nullptr) {
              g0 *= __uint_as_float(wv[j] << 16);
              g1 *= __uint_as_float(wv[j] & 0xffff0000u);
            }
            ov[j] = pack_bf16x2(r * g0 - x0 * c, r * g1 - x1 * c);
          } else {
            const float x0 = __uint_as_float(xv[j]);
            float g0 = __uint_as_float(gv[j]);
            if (w != nullptr) g0 *= __uint_as_float(wv[j]);
            ov[j] = __float_as_uint(r * g0 - x0 * c);
          }
        }
        *reinterpret_cast<u32x4*>(outr + d) = ov;
      }
    } else {
      for (int d = lane; d < D; d += 64) {
        const float x0 = Elem<T>::load(xr + d);
        float g0 = Elem<T>::load(gr + d);
        if (w != nullptr) g0 *= Elem<T>::load(w + d);
        Elem<T>::store(outr + d, r * g0 - x0 * c);
      }
    }
  }
}

// Rows and weight gradient in one pass, for rows of at most NC chunks of 64 x 16 bytes that a wave keeps in registers:
// a block owns a run of rows (its eight waves every eighth of it), a lane adds up dy x r of its columns over its
// wave's rows in ascending order, and at the end the eight waves' sums meet in LDS, a chunk at a time, in the waves'
// order.  partial [gridDim.x][D] f32 (may be null).  dx is rms_norm_backward_rows_kernel's.
//
// A kernel of its own for the weight reads x and dy again, on as many blocks as there are slabs: with the rows' 17.4 us
// at 640 rows of 1024 (20 blocks), 27.2 at 4096 of 2048 (128); together 4.8 and 13.4.
template <typename T, int NC>
__global__ __launch_bounds__(512) void rms_norm_backward_kernel(
    const T* __restrict__ x, const T* __restrict__ w, float eps, const T* __restrict__ dy, int rows, int D,
    T* __restrict__ dx, float* __restrict__ partial) {
  constexpr int VEC = 16 / sizeof(T), COLS = 64 * VEC, WAVES = 8;
  __shared__ __attribute__((aligned(16))) float s_sum[2][WAVES][COLS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float inv_d = 1.0f / (float)D;
  const int per = (rows + (int)gridDim.x - 1) / (int)gridDim.x;
  const int64_t first = (int64_t)blockIdx.x * per;
  const int t1 = (int)(first + per < rows ? first + per : rows);
  auto get = [](u32x4 v, int j) {  // element j of 16 bytes
    if constexpr (sizeof(T) == 2)
      return j & 1 ? __uint_as_float(v[j >> 1] & 0xffff0000u) : __uint_as_float(v[j >> 1] << 16);
    else
      return __uint_as_float(v[j]);
  };
  const u32x4 zero = {0u, 0u, 0u, 0u};
  u32x4 wv[NC];
  float acc[NC][VEC];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int d = i * COLS + lane * VEC;
    wv[i] = w != nullptr && d < D ? *reinterpret_cast<const u32x4*>(w + d) : zero;
#pragma unroll
    for (int j = 0; j < VEC; ++j) acc[i][j] = 0.f;
  }
  for (int64_t t = first + wave; t < t1; t += WAVES) {
    const T* xr = x + (size_t)t * D;
    const T* gr = dy + (size_t)t * D;
    T* outr = dx + (size_t)t * D;
    u32x4 xv[NC], gv[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int d = i * COLS + lane * VEC;
      xv[i] = d < D ? *reinterpret_cast<const u32x4*>(xr + d) : zero;
      gv[i] = d < D ? *reinterpret_cast<const u32x4*>(gr + d) : zero;
    }
    float ss = 0.f, sg = 0.f;
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        const float x0 = get(xv[i], j);
        float g0 = get(gv[i], j);
        if (w != nullptr) g0 *= get(wv[i], j);
        ss += x0 * x0;
        sg += g0 * x0;
      }
    const float r = 1.0f / sqrtf(wave_sum_f32(ss) * inv_d + eps);
    const float c = r * r * r * wave_sum_f32(sg) * inv_d;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      // (the row stays as 16 bits an element: the compiler would keep what it has unpacked, and spill)
      asm volatile("" : "+v"(xv[i]), "+v"(gv[i]), "+v"(wv[i]));
      float o[VEC];
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        const float x0 = get(xv[i], j), dy0 = get(gv[i], j);
        const float g0 = w != nullptr ? dy0 * get(wv[i], j) : dy0;
        o[j] = r * g0 - x0 * c;
        acc[i][j] += dy0 * x0 * r;
      }
      u32x4 ov;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (sizeof(T) == 2) ov[j] = pack_bf16x2(o[2 * j], o[2 * j + 1]);
        else ov[j] = __float_as_uint(o[j]);
      }
      const int d = i * COLS + lane * VEC;
      if (d < D) *reinterpret_cast<u32x4*>(outr + d) = ov;
    }
  }
  if (partial == nullptr) return;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
#pragma unroll
    for (int j = 0; j < VEC; j += 4)
      *reinterpret_cast<f32x4*>(&s_sum[i & 1][wave][lane * VEC + j]) =
          f32x4{acc[i][j], acc[i][j + 1], acc[i][j + 2], acc[i][j + 3]};
    __syncthreads();  // (two buffers: chunk i + 2 is written after the barrier of chunk i + 1, behind every read of i)
    const int d = i * COLS + tid;
    if (tid < COLS && d < D) {
      float sum = s_sum[i & 1][0][tid];
#pragma unroll
      for (int v = 1; v < WAVES; ++v) sum += s_sum[i & 1][v][tid];
      partial[(size_t)blockIdx.x * D + d] = sum;
    }
  }
}

// Longer rows and rows of no whole 16 bytes: the weight gradient, first half.  The rows are cut into gridDim.y slabs; a thread owns 16 bytes' worth
// of columns (one column when D does not divide that way) and adds up dy x r over the rows of its
// slab in ascending order.  partial [slabs][D] f32.
template <typename T>
__global__ __launch_bounds__(256) void rms_norm_backward_weight_kernel(
    const T* __restrict__ x, const T* __restrict__ dy, const float* __restrict__ rstd, int rows,
    int D, float* __restrict__ partial) {
  constexpr int VEC = 16 / sizeof(T);
  const bool vec = D % VEC == 0;
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= (vec ? D / VEC : D)) return;
  const int per = (rows + gridDim.y - 1) / gridDim.y;
  const int t0 = blockIdx.y * per;
  const int t1 = t0 + per < rows ? t0 + per : rows;
  float* out = partial + (size_t)blockIdx.y * D;
  if (vec) {
    float acc[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) acc[j] = 0.f;
#pragma unroll 4
    for (int t = t0; t < t1; ++t) {
      const u32x4 xv = *reinterpret_cast<const u32x4*>(x + (size_t)t * D + c * VEC);
      const u32x4 gv = *reinterpret_cast<const u32x4*>(dy + (size_t)t * D + c * VEC);
      const float r = rstd[t];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (sizeof(T) == 2) {
          acc[2 * j] += __uint_as_float(gv[j] << 16) * __uint_as_float(xv[j] << 16) * r;
          acc[2 * j + 1] += __uint_as_float(gv[j] & 0xffff0000u) * __uint_as_float(xv[j] & 0xffff0000u) * r;
        } else {
          acc[j] += __uint_as_float(gv[j]) * __uint_as_float(xv[j]) * r;
        }
      }
    }
#pragma unroll
    for (int j = 0; j < VEC; ++j) out[c * VEC + j] = acc[j];
  } else {
    float acc = 0.f;
    for (int t = t0; t < t1; ++t)
      acc += Elem<T>::load(dy + (size_t)t * D + c) * Elem<T>::load(x + (size_t)t * D + c) * rstd[t];
    out[c] = acc;
  }
}

// Second half: a block owns 32 columns; its eight groups of 32 threads add every eighth slab in
// ascending order, then the eight sums are added in order.  One rounding.
template <typename T>
__global__ __launch_bounds__(256) void rms_norm_backward_weight_sum_kernel(
    const float* __restrict__ partial, int slabs, int D, T* __restrict__ dw) {
  __shared__ float s_sum[8][32];
  const int col = blockIdx.x * 32 + (threadIdx.x & 31), grp = threadIdx.x >> 5;
  float acc = 0.f;
  if (col < D) {
#pragma unroll 8
    for (int s = grp; s < slabs; s += 8) acc += partial[(size_t)s * D + col];
  }
  s_sum[grp][threadIdx.x & 31] = acc;
  __syncthreads();
  if (grp == 0 && col < D) {
    float total = 0.f;
#pragma unroll
    for (int q = 0; q < 8; ++q) total += s_sum[q][threadIdx.x];
    Elem<T>::store(dw + col, total);
  }
}

// --------------------------------------------------------------------------------- router backward
// One wave per token: dw [K] -> dlogits [E] (zero where the score function does not reach).
//   sigmoid:              w_k = s_k,            s = sigmoid(l_k)    dl_k = dw_k s_k (1 - s_k)
//   sigmoid, renormalised w_k = s_k / S,        S = sum_sel s       dl_k = (dw_k - <dw, w>) / S * s_k (1 - s_k)
//   softmax:              w_k = p_k,            p = softmax(l)      dl_e = p_e ([e selected] dw_e - <dw, w>)
//   softmax, renormalised w_k = p_k / sum_sel p                     dl_k = w_k (dw_k - <dw, w>)
template <typename T>
__global__ __launch_bounds__(256) void router_backward_kernel(
    const float* __restrict__ logits, const int32_t* __restrict__ topk_idx,
    const float* __restrict__ topk_w, const float* __restrict__ d_w, int Tn, int E, int K,
    int score_fn, int renormalize, T* __restrict__ dlogits, int ld) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= Tn) return;
  const int lane = threadIdx.x & 63;
  const float* l = logits + (size_t)t * E;
  // <dw, w> over the selected experts
  float dot = 0.f;
  for (int k = 0; k < K; ++k) dot += d_w[(size_t)t * K + k] * topk_w[(size_t)t * K + k];
  float mx = -INFINITY, den = 0.f, ssum = 0.f;
  if (score_fn == FS2MOE_SCORE_SOFTMAX && !renormalize) {
    for (int e = lane; e < E; e += 64) mx = fmaxf(mx, l[e]);
    // wave-wide maximum through the order-preserving unsigned key of a float
    {
      const uint32_t u = __float_as_uint(mx);
      const uint32_t key = wave_max_u32((u & 0x80000000u) ? ~u : (u | 0x80000000u));
      mx = __uint_as_float((key & 0x80000000u) ? (key & 0x7fffffffu) : ~key);
    }
    for (int e = lane; e < E; e += 64) den += __expf(l[e] - mx);
    den = wave_sum_f32(den);
  }
  if (score_fn == FS2MOE_SCORE_SIGMOID && renormalize) {
    for (int k = 0; k < K; ++k) {
      // an id outside [0, E) selects nothing (the forward stages drop such a pair)
      const int id = topk_idx[(size_t)t * K + k];
      if (id < 0 || id >= E) continue;
      ssum += 1.0f / (1.0f + __expf(-l[id]));
    }
  }
  for (int e = lane; e < E; e += 64) {
    float dw = 0.f, w = 0.f;
    bool sel = false;
    for (int k = 0; k < K; ++k)
      if (topk_idx[(size_t)t * K + k] == e) {
        dw = d_w[(size_t)t * K + k];
        w = topk_w[(size_t)t * K + k];
        sel = true;
      }
    float dl = 0.f;
    if (score_fn == FS2MOE_SCORE_SIGMOID) {
      if (sel) {
        const float s = 1.0f / (1.0f + __expf(-l[e]));
        dl = renormalize ? (dw - dot) / ssum * s * (1.0f - s) : dw * s * (1.0f - s);
      }
    } else if (renormalize) {
      if (sel) dl = w * (dw - dot);
    } else {
      const float p = __expf(l[e] - mx) / den;
      dl = p * ((sel ? dw : 0.f) - dot);
    }
    Elem<T>::store(dlogits + (size_t)t * ld + e, dl);
  }
  for (int e = E + lane; e < ld; e += 64) Elem<T>::store(dlogits + (size_t)t * ld + e, 0.f);
}

}  // namespace fs2moe

using namespace fs2moe;

// One group with fewer tiles than the chip has CUs: the rows are cut into this many segments.
static int wgrad_segments(int64_t rows, int M, int N) {
  const int64_t tiles = (int64_t)((M + wgk::TM - 1) / wgk::TM) * ((N + wgk::TN - 1) / wgk::TN);
  if (tiles >= 128) return 1;
  int64_t s = 256 / tiles;
  const int64_t most = rows / 256;  // at least 256 rows per segment
  s = s < most ? s : most;
  return s >= 2 ? (int)s : 1;
}

// (the f32 tiles are smaller: enough segments for two blocks to a CU)
static int wgrad_segments_f32(int64_t rows, int M, int N) {
  const int64_t tiles = (int64_t)((M + 63) / 64) * ((N + 63) / 64), enough = (511 + tiles) / tiles;
  const int segments = wgrad_segments(rows, M, N);
  return segments < enough ? segments : (int)enough;
}

// A gradient is written once and not read here, and as ordinary stores its lines push the operands' rows,
// which other tiles read again, out of L2: 128 experts of 256 rows, 2048 x 768, 207 us with ordinary and
// 186 us with non-temporal stores (bf16); 8 of 71 rows, 4288 x 5504, 108 and 97.  But rows that do not begin on a
// 128-byte line leave every piece of 128 bytes in two lines, whose halves L2 puts together unless they are marked
// non-temporal: 8 of 71, 4288 x 5496, 131 us with ordinary and 221 with non-temporal stores; 8 of 40, 4096 x 14344,
// 301 and 596; 64 of 220, 2880 x 808, 149 and 173; 128 of 256, 2048 x 776, 254 and 263; 8 of 2048, 4096 x 14344, 1785
// and 1844; 16 of 375, 1024 x 1368, 43 and 50.
static int nt_stores(int64_t N) { return N % 64 == 0; }

// Rows of each of (at most) *segments segments, a multiple of 16; *segments becomes how many that makes,
// none of them empty.
static int segment_rows(int64_t rows, int* segments) {
  const int64_t per = ((rows + *segments - 1) / *segments + 15) / 16 * 16;
  if (rows > 0) *segments = (int)((rows + per - 1) / per);
  return (int)per;
}

static int launch_wgrad_reduce(const float* partial, int segments, int64_t n, int dtype, void* dw,
                               hipStream_t st) {
  const unsigned blocks = (unsigned)((n / 4 + 255) / 256);
  if (dtype == FS2MOE_BF16)
    hipLaunchKernelGGL(wgrad_reduce_kernel<uint16_t>, dim3(blocks), dim3(256), 0, st, partial, segments, n,
                       static_cast<uint16_t*>(dw));
  else
    hipLaunchKernelGGL(wgrad_reduce_kernel<float>, dim3(blocks), dim3(256), 0, st, partial, segments, n,
                       static_cast<float*>(dw));
  return check_launch("wgrad_reduce");
}

// The f32 gradients of one call, in one launch.
static int launch_wgrad_f32(F32WgradJobs& jobs, const int32_t* a_map, const int32_t* counts, const int32_t* offsets, int E,
                            hipStream_t st) {
  int64_t blocks = 0;
  for (int i = 0; i < jobs.n; ++i) {
    F32WgradJob& j = jobs.job[i];
    j.m_tiles = (j.M + 63) / 64;
    j.n_tiles = (j.N + 63) / 64;
    j.first = (int)blocks;
    blocks += (int64_t)(j.grouped ? E : j.segments) * j.m_tiles * j.n_tiles;
    FS2_REQUIRE(blocks <= 0x7fffffffll, "grouped_wgrad: too many tiles");
  }
  const Groups g{counts, offsets, E, 0};
  auto k = a_map != nullptr ? grouped_wgrad_f32_kernel<true> : grouped_wgrad_f32_kernel<false>;
  hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(f32t::threads(1)), 0, st, jobs, a_map, g);
  return check_launch("grouped_wgrad");
}

// One launch for all gradients of `jobs`; the grouped ones share counts and offsets.
static int launch_wgrad(const WgradJobs& jobs, const int32_t* row_map, const int32_t* counts,
                        const int32_t* offsets, int E, hipStream_t st) {
  for (int i = 0; i < jobs.n; ++i) {
    const WgradJob& j = jobs.job[i];
    FS2_REQUIRE((int64_t)(j.M < wgk::TM ? j.M : wgk::TM) * j.N * 2 <= 0xfffffff0ll,
                "grouped_wgrad: M=%d, N=%d: rows of a tile are addressed with 32-bit byte offsets", j.M, j.N);
  }
  auto k = row_map != nullptr ? grouped_wgrad_kernel<true> : grouped_wgrad_kernel<false>;
  static bool attr_set = false;  // benign race: setting the attribute is idempotent
  if (!attr_set) {
    for (const void* p : {reinterpret_cast<const void*>(grouped_wgrad_kernel<false>),
                          reinterpret_cast<const void*>(grouped_wgrad_kernel<true>)}) {
      hipError_t e = hipFuncSetAttribute(p, hipFuncAttributeMaxDynamicSharedMemorySize, wgk::SMEM_BYTES);
      if (e != hipSuccess) {
        set_error("grouped_wgrad: cannot reserve %d bytes of LDS: %s", wgk::SMEM_BYTES, hipGetErrorString(e));
        return FS2MOE_ERR_LAUNCH;
      }
    }
    attr_set = true;
  }
  const int cus = cu_count_by_xcd(), blocks = cus < wgk::MAX_BLOCKS ? cus : wgk::MAX_BLOCKS;
  if (blocks == 0) {
    set_error("grouped_wgrad: cannot query the compute-unit count");
    return FS2MOE_ERR_LAUNCH;
  }
  hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(wgk::WAVES * 64), wgk::SMEM_BYTES, st, jobs, row_map,
                     counts, offsets, E);
  return check_launch("grouped_wgrad");
}

extern "C" int64_t fs2moe_grouped_wgrad_workspace_bytes(int32_t grouped, int32_t M, int32_t N,
                                                        int64_t max_rows) {
  if (M < 1 || N < 1 || max_rows < 0) return -1;
  if (grouped) return 0;
  const int s = wgrad_segments(max_rows, M, N);
  return s > 1 ? (int64_t)s * M * N * 4 : 0;
}

extern "C" int fs2moe_grouped_wgrad(const void* a, const int32_t* a_row_map, const void* b,
                                    const int32_t* counts, const int32_t* offsets, int32_t E,
                                    int32_t M, int32_t N, int64_t max_rows, int32_t dtype, void* dw,
                                    void* workspace, int64_t workspace_bytes, void* stream) {
  FS2_REQUIRE(a && b && dw, "grouped_wgrad: null pointer");
  FS2_REQUIRE((counts == nullptr) == (offsets == nullptr), "grouped_wgrad: counts without offsets");
  FS2_REQUIRE(E >= 1 && E <= FS2MOE_MAX_EXPERTS && (counts != nullptr || E == 1),
              "grouped_wgrad: E=%d", E);
  FS2_REQUIRE(dtype == FS2MOE_F32 || dtype == FS2MOE_BF16, "grouped_wgrad: dtype %d", dtype);
  const int vec = dtype == FS2MOE_BF16 ? 8 : 4;
  FS2_REQUIRE(M > 0 && N > 0 && M % vec == 0 && N % vec == 0,
              "grouped_wgrad: M=%d and N=%d must be positive multiples of %d", M, N, vec);
  FS2_REQUIRE(max_rows >= 0 && max_rows < (1ll << 31), "grouped_wgrad: max_rows=%lld",
              (long long)max_rows);
  FS2_REQUIRE(aligned16(a) && aligned16(b) && aligned16(dw) && aligned16(workspace),
              "grouped_wgrad: buffers must be 16-byte aligned");
  const int m_tiles = (M + wgk::TM - 1) / wgk::TM, n_tiles = (N + wgk::TN - 1) / wgk::TN;
  // one group: segments of its rows (each a slot of the grid) when there is scratch for their sums
  int segments = 1;
  if (counts == nullptr) {
    segments = dtype == FS2MOE_F32 ? wgrad_segments_f32(max_rows, M, N) : wgrad_segments(max_rows, M, N);
    if (workspace == nullptr || workspace_bytes < (int64_t)segments * M * N * 4) segments = 1;
  }
  const int seg_rows = segment_rows(max_rows, &segments);
  const int slots = counts != nullptr ? E : segments;
  float* partial = segments > 1 ? static_cast<float*>(workspace) : nullptr;
  FS2_REQUIRE((int64_t)slots * m_tiles * n_tiles <= 0x7fffffffll, "grouped_wgrad: too many tiles");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool mapped = a_row_map != nullptr;
  if (dtype == FS2MOE_BF16) {
    WgradJobs jobs;
    jobs.n = 1;
    jobs.job[0] = {static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(b),
                   static_cast<uint16_t*>(dw), partial, M, N, m_tiles, m_tiles * n_tiles,
                   counts != nullptr, slots, seg_rows, (int)max_rows, nt_stores(N), mapped, 0};
    // (without rows nothing is read, and the map may be empty)
    if (int rc = launch_wgrad(jobs, max_rows > 0 ? a_row_map : nullptr, counts, offsets, E, st)) return rc;
  } else {
    F32WgradJobs jobs;
    jobs.n = 1;
    jobs.job[0] = {static_cast<const float*>(a), static_cast<const float*>(b), static_cast<float*>(dw), partial, M, N, 0, 0,
                   segments, seg_rows, (int)max_rows, counts != nullptr, 0};
    if (int rc = launch_wgrad_f32(jobs, a_row_map, counts, offsets, E, st)) return rc;
  }
  return segments > 1 ? launch_wgrad_reduce(partial, segments, (int64_t)M * N, dtype, dw, st) : FS2MOE_OK;
}

// The CUs that a plan counts on.  A constant and not the device's own number, which the launch asks for: a plan
// sizes scratch in calls that touch no device, and must come out the same when it is launched.  With other
// numbers of CUs (a partition of the chip) its cuts are only less even.
constexpr int kPlanCUs = 256;

int64_t fs2moe::wgrad_plan(WgradRequest* r, int n, int32_t E, int64_t planned, int64_t rows,
                           int32_t dtype) {
  if (dtype == FS2MOE_F32) {  // every single group is cut as in fs2moe_grouped_wgrad
    int64_t bytes = 0;
    for (int i = 0; i < n; ++i) {
      r[i].segments = r[i].grouped ? 1 : wgrad_segments_f32(rows, r[i].M, r[i].N);
      if (r[i].segments > 1) bytes += (int64_t)r[i].segments * r[i].M * r[i].N * 4;
    }
    return bytes;
  }
  auto tiles = [](const WgradRequest& q) {
    return (int64_t)((q.M + wgk::TM - 1) / wgk::TM) * ((q.N + wgk::TN - 1) / wgk::TN);
  };
  const int64_t one = rows / wgk::RK + wgk::kTileCost;
  int64_t total = 0;
  for (int i = 0; i < n; ++i)
    total += tiles(r[i]) * (r[i].grouped ? planned / wgk::RK + (int64_t)E * wgk::kTileCost : one);
  const int64_t fair = total / kPlanCUs + 1;
  int64_t bytes = 0;
  for (int i = 0; i < n; ++i) {
    r[i].segments = 1;
    if (r[i].grouped || one <= fair) continue;
    // at least 256 rows each, and no more than gives every CU a tile of this gradient
    int64_t s = (one + fair - 1) / fair;
    const int64_t by_rows = rows / 256, by_cus = kPlanCUs / tiles(r[i]) + 1;
    s = s < by_rows ? s : by_rows;
    s = s < by_cus ? s : by_cus;
    if (s < 2) continue;
    r[i].segments = (int)s;
    bytes += s * r[i].M * r[i].N * 4;
  }
  return bytes;
}

int fs2moe::wgrad_all(const WgradRequest* r, int n, const int32_t* row_map, const int32_t* counts,
                      const int32_t* offsets, int32_t E, int64_t grouped_rows, int64_t rows, int32_t dtype,
                      void* scratch, void* stream) {
  if (dtype == FS2MOE_F32) {
    F32WgradJobs jobs;
    FS2_REQUIRE(n <= F32WgradJobs::MAX, "wgrad: internal: %d gradients", n);
    jobs.n = 0;
    float* part = static_cast<float*>(scratch);
    // (those of one group first: their segments are the longer walks)
    for (const bool grouped : {false, true})
      for (int i = 0; i < n; ++i) {
        const WgradRequest& q = r[i];
        if (q.grouped != grouped) continue;
        int segments = grouped ? 1 : q.segments;
        const int seg = segment_rows(rows, &segments);
        jobs.job[jobs.n] = {static_cast<const float*>(q.a), static_cast<const float*>(q.b), static_cast<float*>(q.dw),
                            segments > 1 ? part : nullptr, q.M, q.N, 0, 0, segments, seg, (int)rows, grouped, 0};
        if (segments > 1) part += (int64_t)segments * q.M * q.N;
        ++jobs.n;
      }
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (int rc = launch_wgrad_f32(jobs, nullptr, counts, offsets, E, st)) return rc;
    for (int i = 0; i < jobs.n; ++i) {
      const F32WgradJob& j = jobs.job[i];
      if (j.partial != nullptr)
        if (int rc = launch_wgrad_reduce(j.partial, j.segments, (int64_t)j.M * j.N, dtype, j.C, st)) return rc;
    }
    return FS2MOE_OK;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  FS2_REQUIRE(n <= wgk::MAX_JOBS, "wgrad: internal: %d gradients", n);
  WgradJobs jobs;
  jobs.n = n;
  float* part = static_cast<float*>(scratch);
  bool any_grouped = false, any_mapped = false;
  for (int i = 0; i < n; ++i) {
    const WgradRequest& q = r[i];
    const int mt = (q.M + wgk::TM - 1) / wgk::TM, nt = (q.N + wgk::TN - 1) / wgk::TN;
    any_grouped = any_grouped || q.grouped;
    any_mapped = any_mapped || q.map_a || q.map_b;
    int segments = q.grouped ? 1 : q.segments;
    const int seg = segment_rows(rows, &segments), slots = q.grouped ? E : segments;
    jobs.job[i] = {static_cast<const uint16_t*>(q.a), static_cast<const uint16_t*>(q.b),
                   static_cast<uint16_t*>(q.dw), !q.grouped && slots > 1 ? part : nullptr, q.M, q.N, mt, mt * nt,
                   q.grouped ? 1 : 0, slots, q.grouped ? 0 : seg, (int)rows, nt_stores(q.N),
                   q.map_a, q.map_b};
    if (!q.grouped && slots > 1) part += (int64_t)slots * q.M * q.N;
  }
  if (int rc = launch_wgrad(jobs, any_mapped ? row_map : nullptr, any_grouped ? counts : nullptr,
                            any_grouped ? offsets : nullptr, any_grouped ? E : 0, st))
    return rc;
  for (int i = 0; i < n; ++i)
    if (jobs.job[i].partial != nullptr)
      if (int rc = launch_wgrad_reduce(jobs.job[i].partial, jobs.job[i].slots, (int64_t)r[i].M * r[i].N, dtype,
                                       r[i].dw, st))
        return rc;
  return FS2MOE_OK;
}

extern "C" int fs2moe_swiglu_backward(const void* g, const void* u, const void* dh, int64_t rows,
                                      int32_t F, int32_t dtype, void* h, void* dg, void* du,
                                      void* stream) {
  FS2_REQUIRE(g && u && dh && h && dg && du, "swiglu_backward: null pointer");
  FS2_REQUIRE(dtype == FS2MOE_F32 || dtype == FS2MOE_BF16, "swiglu_backward: dtype %d", dtype);
  FS2_REQUIRE(rows >= 0 && F > 0 && F % 8 == 0, "swiglu_backward: rows=%lld, F=%d",
              (long long)rows, F);
  FS2_REQUIRE(aligned16(g) && aligned16(u) && aligned16(dh) && aligned16(h) && aligned16(dg) &&
                  aligned16(du),
              "swiglu_backward: buffers must be 16-byte aligned");
  const int64_t n = rows * F;
  if (n == 0) return FS2MOE_OK;
  const int vec = dtype == FS2MOE_BF16 ? 8 : 4;
  int64_t blocks = (n / vec + 255) / 256;
  if (blocks > 16384) blocks = 16384;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == FS2MOE_BF16)
    hipLaunchKernelGGL(swiglu_backward_kernel<uint16_t>, dim3((unsigned)blocks), dim3(256), 0, st,
                       static_cast<const uint16_t*>(g), static_cast<const uint16_t*>(u),
                       static_cast<const uint16_t*>(dh), n, static_cast<uint16_t*>(h),
                       static_cast<uint16_t*>(dg), static_cast<uint16_t*>(du));
  else
    hipLaunchKernelGGL(swiglu_backward_kernel<float>, dim3((unsigned)blocks), dim3(256), 0, st,
                       static_cast<const float*>(g), static_cast<const float*>(u),
                       static_cast<const float*>(dh), n, static_cast<float*>(h),
                       static_cast<float*>(dg), static_cast<float*>(du));
  return check_launch("swiglu_backward");
}

extern "C" int fs2moe_pair_dot(const void* a, const void* a2, const int32_t* a_rows, const void* b,
                               int32_t T, int32_t K, int32_t D, int32_t dtype, float* out,
                               void* stream) {
  FS2_REQUIRE(a && a_rows && b && out, "pair_dot: null pointer");
  FS2_REQUIRE(dtype == FS2MOE_F32 || dtype == FS2MOE_BF16, "pair_dot: dtype %d", dtype);
  FS2_REQUIRE(T >= 0 && K >= 1 && K <= FS2MOE_MAX_TOP_K && D > 0, "pair_dot: T=%d, K=%d, D=%d", T, K,
              D);
  const int64_t pairs = (int64_t)T * K;
  FS2_REQUIRE(pairs < (1ll << 31), "pair_dot: too many pairs");
  if (pairs == 0) return FS2MOE_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const unsigned blocks = (unsigned)((pairs + 3) / 4);
  // 16-byte loads need rows that start on 16 bytes: D a multiple of the vector and aligned bases
  const int vec = 16 / elem_size(dtype);
  const int vec_ok = D % vec == 0 && aligned16(a) && aligned16(b) && (a2 == nullptr || aligned16(a2));
  if (dtype == FS2MOE_BF16)
    hipLaunchKernelGGL(pair_dot_kernel<uint16_t>, dim3(blocks), dim3(256), 0, st,
                       static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(a2), a_rows,
                       static_cast<const uint16_t*>(b), (int)pairs, K, D, vec_ok, out);
  else
    hipLaunchKernelGGL(pair_dot_kernel<float>, dim3(blocks), dim3(256), 0, st,
                       static_cast<const float*>(a), static_cast<const float*>(a2), a_rows,
                       static_cast<const float*>(b), (int)pairs, K, D, vec_ok, out);
  return check_launch("pair_dot");
}

extern "C" int fs2moe_router_backward(const float* logits, const int32_t* topk_idx,
                                      const float* topk_w, const float* d_w, int32_t T, int32_t E,
                                      int32_t K, int32_t score_fn, int32_t renormalize,
                                      int32_t dtype, void* dlogits, void* stream) {
  FS2_REQUIRE(logits && topk_idx && topk_w && d_w && dlogits, "router_backward: null pointer");
  FS2_REQUIRE(dtype == FS2MOE_F32 || dtype == FS2MOE_BF16, "router_backward: dtype %d", dtype);
  FS2_REQUIRE(T >= 0 && E >= 1 && E <= FS2MOE_MAX_EXPERTS && K >= 1 && K <= FS2MOE_MAX_TOP_K &&
                  K <= E,
              "router_backward: T=%d, E=%d, K=%d", T, E, K);
  FS2_REQUIRE(score_fn == FS2MOE_SCORE_SIGMOID || score_fn == FS2MOE_SCORE_SOFTMAX,
              "router_backward: score_fn %d", score_fn);
  if (T == 0) return FS2MOE_OK;
  return router_backward_ld(logits, topk_idx, topk_w, d_w, T, E, K, score_fn, renormalize, dtype, dlogits, E,
                            stream);
}

int fs2moe::router_backward_ld(const float* logits, const int32_t* topk_idx, const float* topk_w,
                               const float* d_w, int32_t T, int32_t E, int32_t K, int32_t score_fn,
                               int32_t renormalize, int32_t dtype, void* dlogits, int32_t ld,
                               void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  const unsigned blocks = (unsigned)((T + 3) / 4);
  if (dtype == FS2MOE_BF16)
    hipLaunchKernelGGL(router_backward_kernel<uint16_t>, dim3(blocks), dim3(256), 0, st, logits,
                       topk_idx, topk_w, d_w, T, E, K, score_fn, renormalize,
                       static_cast<uint16_t*>(dlogits), ld);
  else
    hipLaunchKernelGGL(router_backward_kernel<float>, dim3(blocks), dim3(256), 0, st, logits,
                       topk_idx, topk_w, d_w, T, E, K, score_fn, renormalize,
                       static_cast<float*>(dlogits), ld);
  return check_launch("router_backward");
}

// slabs of rows for the weight gradient of the normalisation: eight rows each (a row for each of a block's waves), at
// most 256
static int norm_weight_slabs(int64_t rows) {
  const int64_t s = (rows + 7) / 8;
  return s < 1 ? 1 : (s > 256 ? 256 : (int)s);
}

extern "C" int64_t fs2moe_rms_norm_backward_workspace_bytes(int32_t T, int32_t D) {
  if (T < 0 || D < 1) return -1;
  // rstd [T] (padded to 16 bytes), then the slabs' partial sums.  (rstd is for rows past the one pass alone; how long
  // those are depends on the type, which this size does not)
  return ((int64_t)T * 4 + 15) / 16 * 16 + (int64_t)norm_weight_slabs(T) * D * 4;
}

extern "C" int fs2moe_rms_norm_backward(const void* x, const void* weight, float eps,
                                        const void* dy, int32_t T, int32_t D, int32_t dtype,
                                        void* dx, void* dweight, void* workspace,
                                        int64_t workspace_bytes, void* stream) {
  FS2_REQUIRE(x && dy && dx, "rms_norm_backward: null pointer");
  FS2_REQUIRE(dtype == FS2MOE_F32 || dtype == FS2MOE_BF16, "rms_norm_backward: dtype %d", dtype);
  FS2_REQUIRE(T >= 0 && D > 0, "rms_norm_backward: T=%d, D=%d", T, D);
  FS2_REQUIRE(dweight == nullptr || weight != nullptr,
              "rms_norm_backward: a weight gradient without a weight");
  FS2_REQUIRE(dx != dy && dx != x, "rms_norm_backward: dx must not alias x or dy");
  FS2_REQUIRE(aligned16(x) && aligned16(dy) && aligned16(dx) && aligned16(weight) &&
                  aligned16(workspace),
              "rms_norm_backward: buffers must be 16-byte aligned");
  hipStream_t st = static_cast<hipStream_t>(stream);
  float* rstd = nullptr;
  float* partial = nullptr;
  if (dweight != nullptr) {
    FS2_REQUIRE(workspace != nullptr &&
                    workspace_bytes >= fs2moe_rms_norm_backward_workspace_bytes(T, D),
                "rms_norm_backward: the weight gradient needs a workspace of %lld bytes",
                (long long)fs2moe_rms_norm_backward_workspace_bytes(T, D));
    rstd = static_cast<float*>(workspace);
    partial = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) +
                                       ((int64_t)T * 4 + 15) / 16 * 16);
  }
  const int slabs = norm_weight_slabs(T);
  const int vec = dtype == FS2MOE_BF16 ? 8 : 4;
  const int chunks = D % vec == 0 ? (D / vec + 63) / 64 : 0;
  // (rows whose 16-byte pieces and sums a lane holds in its registers: D up to 4096 in bf16, 2560 in f32.  With ten
  // pieces in bf16 they spill: 2000 rows of 5120 40.1 us, the kernels of their own 28.1)
  const bool one_pass = T > 0 && chunks >= 1 && chunks <= (dtype == FS2MOE_BF16 ? 8 : 10);
  if (one_pass) {
    auto launch = [&](auto type, auto nc) {
      using E = decltype(type);
      hipLaunchKernelGGL((rms_norm_backward_kernel<E, decltype(nc)::value>), dim3((unsigned)slabs), dim3(512), 0, st,
                         static_cast<const E*>(x), static_cast<const E*>(weight), eps, static_cast<const E*>(dy), T, D,
                         static_cast<E*>(dx), partial);
    };
    auto by_chunks = [&](auto type) {
      if (chunks <= 1) launch(type, std::integral_constant<int, 1>{});
      else if (chunks <= 2) launch(type, std::integral_constant<int, 2>{});
      else if (chunks <= 4) launch(type, std::integral_constant<int, 4>{});
      else if (chunks <= 6) launch(type, std::integral_constant<int, 6>{});
      else launch(type, std::integral_constant<int, sizeof(type) == 2 ? 8 : 10>{});
    };
    if (dtype == FS2MOE_BF16) by_chunks(uint16_t{});
    else by_chunks(float{});
    if (int rc = check_launch("rms_norm_backward")) return rc;
  } else if (T > 0) {
    int blocks = (T + 3) / 4;
    if (blocks > 4096) blocks = 4096;
    if (dtype == FS2MOE_BF16)
      hipLaunchKernelGGL(rms_norm_backward_rows_kernel<uint16_t>, dim3((unsigned)blocks), dim3(256),
                         0, st, static_cast<const uint16_t*>(x),
                         static_cast<const uint16_t*>(weight), eps,
                         static_cast<const uint16_t*>(dy), T, D, static_cast<uint16_t*>(dx), rstd);
    else
      hipLaunchKernelGGL(rms_norm_backward_rows_kernel<float>, dim3((unsigned)blocks), dim3(256), 0,
                         st, static_cast<const float*>(x), static_cast<const float*>(weight), eps,
                         static_cast<const float*>(dy), T, D, static_cast<float*>(dx), rstd);
    if (int rc = check_launch("rms_norm_backward")) return rc;
  }
  if (dweight == nullptr) return FS2MOE_OK;
  // (with no rows the one slab sums nothing and the gradient is zero)
  const int owners = D % vec == 0 ? D / vec : D;  // threads per slab
  const dim3 grid((unsigned)((owners + 255) / 256), (unsigned)slabs);
  const unsigned sum_blocks = (unsigned)((D + 31) / 32);
  if (dtype == FS2MOE_BF16) {
    if (!one_pass)
      hipLaunchKernelGGL(rms_norm_backward_weight_kernel<uint16_t>, grid, dim3(256), 0, st,
                       static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(dy), rstd, T, D,
                       partial);
    hipLaunchKernelGGL(rms_norm_backward_weight_sum_kernel<uint16_t>, dim3(sum_blocks), dim3(256), 0, st,
                       partial, slabs, D, static_cast<uint16_t*>(dweight));
  } else {
    if (!one_pass)
      hipLaunchKernelGGL(rms_norm_backward_weight_kernel<float>, grid, dim3(256), 0, st,
                       static_cast<const float*>(x), static_cast<const float*>(dy), rstd, T, D,
                       partial);
    hipLaunchKernelGGL(rms_norm_backward_weight_sum_kernel<float>, dim3(sum_blocks), dim3(256), 0, st,
                       partial, slabs, D, static_cast<float*>(dweight));
  }
  return check_launch("rms_norm_backward (weight)");
}
