// f32 GEMMs of the expert networks and of their backward pass, on v_mfma_f32_32x32x2_f32 (true f32
// products and sums).
//
// What bounds them: the matrix pipe (64 clocks per instruction and SIMD, 157 TFLOP/s nominal, 154 in a
// large product of the vendor's library), and, with few tiles, their number against 256 CUs.  A chunk is
// 32 k; two chunks are on their way from memory in two register sets while a third is multiplied, LDS
// holds two (one barrier per chunk), and a block is 4 waves (or 8) on a 64 x 64, 4 on a 32 x 64 or 4 on a 128 x 128 tile,
// several of the smaller ones' blocks to a CU (f32t::large_tiles, flat_tiles).  What a
// wave does besides multiplying is dealt out one instruction behind each product (Walk::run): as phases,
// i.e. stores, barrier, loads, reads, products, the same tiles reach 132 TFLOP/s with every SIMD full
// and 95 with one wave on each, whether one chunk or four are in flight; dealt out 149-154 and 107.
// 8192 x 2048 by 2048 x 4096: 1012 -> 949 us (the library's product 923); the kernels before these, 64 x 64
// tiles of 16 k one chunk ahead and 256 x 256 tiles for the weight gradients: 512 x 1408 by 8 experts of
// 250 rows on average 52 -> 36 us a product and 83 -> 28 us a weight gradient.
//
// k slots.  Lanes 0..31 carry one k of an instruction and lanes 32..63 the other, and which k they are is
// free as long as both operands agree: instruction j of step s takes k 8 s + j and 8 s + 4 + j, so that a
// lane's four values of a k-contiguous operand are one 16-byte LDS read.  Products add the first halves of all chunks
// (steps 0 and 1) in one sum, the second ones (2 and 3) in another, and the two at the end, on every tile: on some
// two groups of waves take a half each, and a row's bits do not depend on the tile.  Two sums of half the length also
// round less (K 1408 4.8e-7 of the result instead of 6.7e-7); on large tiles, which keep both in a wave's registers,
// they take the same time (8192 x 2048 by 2048 x 4096 971, 972 us).
//
// LDS layouts (16-byte chunks).  k-contiguous operand: rows of 128 bytes, chunk c of row r in slot
// c ^ ((r >> 1) & 7).  k-major operand: a row per k, chunk c of row k in slot c ^ (((k >> 2) & 1) << 3), so
// that the two half waves, which read rows 4 apart, use different banks.
#pragma once

#include <type_traits>

#include "common.h"
#include "tile_map.h"

namespace fs2moe {
namespace f32t {
constexpr int BK = 32;
// Threads of a block: four waves, or two groups of four that each take half of every chunk's k, whose sums are added
// at the end.  Two waves to a SIMD cover each other's reads and barriers, and where a tile has up to 32 rows every SIMD
// has one that multiplies: 16 experts of 18 rows, K 1792, N 1024, 38 -> 30 us; 1024 rows, K 4096, N 1024 (a tile a CU)
// 80 -> 74; 60 experts of 80, the pair of D 768, F 2000, 575 -> 547.  Not for two products at once: what the sums leave
// of registers and LDS lets two such blocks share a CU instead of three smaller ones (60 experts of 17 rows, K 576, N
// 1760, 66 -> 80 us).
constexpr int threads(int groups, int wm = 2) { return 128 * wm * groups; }

// Products on tiles of 128 x 128 (two products at once: 128 rows x 64 channels of each) instead of 64 x 64: where their
// rounds of tiles take less time.  In hundredths of a us per 32 k, on full rounds: a small tile 54, of two products 103, a
// large one 195; so full rounds of large ones take a tenth less (two products a twentieth), and whatever part of a last
// round is empty decides most cases.  us, small and large tiles, one product and two:
//   8192 rows, N 2048, K 4096; N 4096, K 2048                 1108, 996; 2116, 1998    (4 and 16 rounds of large ones)
//   8 experts of 2048, the same                               2500, 2379; 4829, 4404
//   4 of 2048, N 1024, K 2048; N 2048, K 1024                  320, 393; 602, 610      (2.1 and 8.3 rounds)
//   8 of 1024, N 2048, K 2048                                  597, 651; 1164, 1169
//   16 of 500, D 768, F 1536, the layer                        521, 539
//   128 of 256, D 1024, F 1024                                 1896, 1971
// rows: the experts' rows, half of a last row block each.  One round of large tiles leaves a SIMD one wave, and few rounds
// of experts' tiles are as uneven as their loads: 8 of 187 rows, D 1024, F 2048, the layer 227, 224 loaded evenly and 227,
// 256 by a popularity law.
// The weight gradients' tiles are small ones.  Large ones give a step up to 2.5 % where their rounds are many and full
// (with the largest experts first, and one gradient up to 15 % by a skewed load) and cost up to 8 % elsewhere; no size
// tells these apart from the load.  us on small and on large tiles, of one gradient and of whole training steps:
//   8192 rows, 2048 x 4096                999, 990       8 experts of 512            554, 548, by a law of 1.2 527, 541
//   8192 rows, 1024 x 2048                277, 510       16 of 500, 1024 x 2048      262, 267                  315, 275
//   64 of 256, 1024 x 1024                296, 304; 331, 407 by a law      32 of 100, 2048 x 2048  319, 381
//   4096 tokens, top-2 of 8, D 1024, F 2048      2615, 2588; by a law of 1.2 2698, 2736
//   4096, top-4 of 64, D 1024, F 1024            2902, 2862                  2923, 2961
//   4096, top-4 of 32, D 1024, F 2048            by laws of 1.1, three of them 5952, 5808; 5827, 5800; 5871, 5819
//   4096, top-8 of 128, D 1024, F 768            4376, 4351; 4633, 4625; 4657, 4644; 4666, 4623
//   4000, top-2 of 16, D 1024, F 2048            by the law 2994, 3038; 2931, 2948; 2934, 3005
//   1500, top-1 of 8, D 1024, F 2048             by the law 663, 715
//   1000, top-2 of 8, D 512, F 1408              365, 385
inline bool large_tiles(bool dual, int64_t rows, int groups, int N, int cus) {
  const int64_t real = groups > 0 && rows > 15ll * groups ? rows - 15ll * groups : rows;  // (less the blocks' padding)
  const int g = groups > 0 ? groups : 1;
  auto blocks = [&](int bm) { return g + (real > (int64_t)g * (bm / 2) ? (real - (int64_t)g * (bm / 2)) / bm : 0); };
  auto rounds = [&](int64_t tiles) { return (tiles + cus - 1) / cus; };
  const int64_t small = rounds(blocks(64) * ((N + 63) / 64)) * (dual ? 103 : 54);
  const int64_t large = rounds(blocks(128) * (dual ? (N + 63) / 64 : (N + 127) / 128));
  return large * 195 < small && large >= (groups == 0 ? 2 : 4);
}

// Where large_tiles says no: products on tiles of 32 x 64 (two groups of two waves), whose rounds are half as long, so that
// what is empty of a last one costs less, and an expert's last row block is half as empty.  In hundredths of a us per 32 k
// on full rounds: 29, of two products 58 (their weights go through LDS for half as many rows).  Experts of up to 32 rows
// have as many tiles of either kind: one product takes the flat ones where a CU has at most one, as the busiest experts
// have two, two products where there are more, since a tile of 64 rows then leaves half of its waves idle.  us on tiles of
// 64 x 64 and on these, the layer and (last) a training step:
//   1000 tokens, top-2 of 8, D 512, F 1408, training          356, 332    (280 tiles on 256 CUs down, 790 gate/up)
//   1000, top-1 of 8, D 1024, F 2048                          188, 171, 496, 482    4000, top-1 of 8, D 576, F 640 340, 329
//   100, top-2 of 8 by a law of 1.1, D 512, F 1408            67.3, 59.1            300, 16, D 768, F 2048 91.9, 80.8
//   64, top-4 of 60, D 1024, F 1024                           200, 185, 653, 639    200, top-6 of 128, D 1024, F 1792 586, 561
// and where the rule says no: gate/up of 1500, top-6 of 64, D 640, F 1728 569, 595; of 2000, top-2 of 8, D 1024, F 1408
// 331, 345; down of 200, top-6 of 128 586, 593.
inline bool flat_tiles(bool dual, int64_t rows, int groups, int N, int parts, int cus) {
  const int64_t real = groups > 0 && rows > 15ll * groups ? rows - 15ll * groups : rows;
  const int g = groups > 0 ? groups : 1;
  const int64_t nt = (int64_t)((N + 63) / 64) * parts;
  if (real <= 32ll * g) return dual ? g * nt > cus : g * nt <= cus;
  auto blocks = [&](int bm) { return g + (real - (int64_t)g * (bm / 2)) / bm; };
  auto rounds = [&](int64_t tiles) { return (tiles + cus - 1) / cus; };
  return rounds(blocks(32) * nt) * (dual ? 58 : 29) < rounds(blocks(64) * nt) * (dual ? 103 : 54);
}

// what a load through a row map reads past the end (not const: a global address)
static __device__ __attribute__((aligned(16))) uint32_t zero16[4] = {0u, 0u, 0u, 0u};

// A chunk (32 k) of one operand: ROWS rows (or columns) x 32 k.  `base` points at the operand's first row
// (column) of the tile in k 0; ld is the stride in floats of a row (k-contiguous) or of a k (k-major).
template <int ROWS, bool KMAJOR, int THREADS>
struct Operand {
  static constexpr int BYTES = ROWS * BK * 4;
  static constexpr int PER = ROWS * BK / 4 / THREADS;  // 16-byte chunks per thread
  static constexpr int CPK = ROWS / 4;                 // k-major: chunks per k
  uint32_t off[PER];
  bool ok[KMAJOR ? PER : 1];  // k-major: the chunk's columns exist

  // rows: how many of the tile's rows (columns) exist, at least 1.  Rows past them repeat the last one
  // (their results are not stored), columns past them are zeros.
  __device__ __forceinline__ void setup(int tid, int ld, int rows) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = tid + THREADS * i;
      if constexpr (KMAJOR) {
        off[i] = (uint32_t)((c / CPK) * ld + (c % CPK) * 4) * 4u;
        ok[i] = (c % CPK) * 4 < rows;
      } else {
        const int r = c >> 3;
        off[i] = (uint32_t)((r < rows ? r : rows - 1) * ld + (c & 7) * 4) * 4u;
      }
    }
  }
  // The pieces of k from k0 on, `left` of them (what lies past the end loads zeros and touches no memory):
  // where they come from, then piece by piece.
  struct From {
    __amdgpu_buffer_rsrc_t rsrc;
    int left;
  };
  static __device__ __forceinline__ From from(const float* base, int ld, int k0, int left) {
    const float* p = KMAJOR ? base + (size_t)k0 * ld : base + k0;
    return From{__builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, 0xfffffff0u, 0x00020000), left};
  }
  __device__ __forceinline__ u32x4 load(const From& f, int tid, int i) const {
    const bool in = KMAJOR ? ok[i] && (tid + THREADS * i) / CPK < f.left : (tid & 7) * 4 < f.left;
    return __builtin_amdgcn_raw_buffer_load_b128(f.rsrc, in ? off[i] : 0xfffffff0u, 0, 0);
  }
  // the same of a k-major operand whose row k is row map[k] of `base`
  __device__ __forceinline__ void load_mapped(u32x4 (&reg)[PER], int tid, const float* base, int ld,
                                              const int32_t* map, int k0, int left) const {
    static_assert(KMAJOR, "the rows of the contraction are mapped");
    int row[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int k = (tid + THREADS * i) / CPK;
      row[i] = map[left > 0 ? k0 + (k < left ? k : left - 1) : 0];
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = tid + THREADS * i;
      const float* p = base + (size_t)row[i] * ld + (c % CPK) * 4;
      if (!(ok[i] && c / CPK < left)) p = reinterpret_cast<const float*>(zero16);
      reg[i] = *reinterpret_cast<const u32x4*>(p);
    }
  }
  static __device__ __forceinline__ void store(u32x4 reg, int tid, int i, uint8_t* lds) {
    const int c = tid + THREADS * i;
    const int at = KMAJOR ? (c / CPK) * CPK + ((c % CPK) ^ (((c / CPK) >> 2 & 1) << 3))
                          : (c >> 3) * 8 + ((c & 7) ^ ((c >> 4) & 7));
    *reinterpret_cast<u32x4*>(lds + at * 16) = reg;
  }
  // the lane's four values of step s (k 8 s + 4 (lane / 32) + 0..3) of the 32 rows from r0 on
  static __device__ __forceinline__ f32x4 frag(const uint8_t* lds, int lane, int r0, int s) {
    const int lr = lane & 31, lk = lane >> 5;
    if constexpr (KMAJOR) {
      const float* p = reinterpret_cast<const float*>(lds) + (8 * s + 4 * lk) * ROWS + ((r0 + lr) ^ (lk << 5));
      return f32x4{p[0], p[ROWS], p[2 * ROWS], p[3 * ROWS]};
    } else {
      const int r = r0 + lr;
      return *reinterpret_cast<const f32x4*>(lds + r * 128 + (((2 * s + lk) ^ ((r >> 1) & 7)) << 4));
    }
  }
};

// The walk over k of one tile: waves WM x 2, each 32 FM rows x 32 FN channels of each of NB matrices.
// acc[b][fn][fm] is the transposed 32 x 32 tile (lane: row lr, channels 8 q + 4 lk + 0..3 in 4 q ..).
// With two sources the second pair follows the first in the same accumulators.
// A_MAPPED: a_map gives the rows of the k-major A.
// HALVES: two sums, over the first and the second half of every chunk's k, added at the end; the groups' (GROUPS 2), or
// both of each wave.
template <int NB, int FM, int FN, bool A_KMAJOR, bool B_KMAJOR, bool A_MAPPED = false, int GROUPS = 1,
          bool HALVES = true, int WM = 2>
struct Walk {
  static_assert(HALVES || GROUPS == 1, "two groups of waves take a half each");
  static constexpr int CHAINS = HALVES && GROUPS == 1 ? 2 : 1;  // sums that a wave keeps
  static constexpr int BM = 32 * WM * FM, BN = 64 * FN, THREADS = threads(GROUPS, WM);
  using OpA = Operand<BM, A_KMAJOR, THREADS>;
  using OpB = Operand<BN, B_KMAJOR, THREADS>;
  static constexpr int BUF_BYTES = OpA::BYTES + NB * OpB::BYTES;
  static constexpr int SMEM_BYTES = 2 * BUF_BYTES;
  static constexpr int PIECES = OpA::PER + NB * OpB::PER;  // 16-byte pieces of a chunk per thread
  static constexpr int STEPS = BK / 8 / GROUPS;              // steps of 8 k of a chunk per wave
  static constexpr int PRODUCTS = 4 * STEPS * NB * FM * FN;  // MFMAs of a chunk per wave

  // The wave's rows and channels of the tile, and which share of a chunk's k it takes.  (Waves w and w + 4 share a
  // SIMD: with a tile of up to 32 rows every SIMD has a wave that multiplies.)
  static __device__ __forceinline__ int wave_m(int wave) { return WM == 1 ? 0 : GROUPS == 2 ? wave >> 2 : wave & 1; }
  static __device__ __forceinline__ int wave_n(int wave) { return WM == 1 || GROUPS == 2 ? wave & 1 : wave >> 1; }
  static __device__ __forceinline__ int wave_group(int wave) { return GROUPS == 2 ? (wave >> 1) & 1 : 0; }

  struct Source {
    const float* a;
    const float* b[NB];
  };
  // m_rows, n_cols: how many of the tile's rows and channels exist; `active`: this wave's rows do.  The walk is the
  // part-th of `parts`, each as many chunks but the last.
  static __device__ __forceinline__ void run(f32x16 (&sums)[NB][FN][FM], uint8_t* smem, const Source& s0,
                                             const Source& s1, int sources, int lda, int ldb, int K,
                                             int m_rows, int n_cols, bool active,
                                             const int32_t* a_map = nullptr, int part = 0, int parts = 1) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave_m(wave), wn = wave_n(wave), s0k = wave_group(wave) * STEPS;
    f32x16 acc[CHAINS][NB][FN][FM];
#pragma unroll
    for (int c = 0; c < CHAINS; ++c)
#pragma unroll
      for (int m = 0; m < NB; ++m)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
#pragma unroll
          for (int fm = 0; fm < FM; ++fm)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[c][m][fn][fm][i] = 0.f;
    OpA opa;
    OpB opb;
    opa.setup(tid, lda, m_rows);
    opb.setup(tid, ldb, n_cols);
    const int nk = (K + BK - 1) / BK, all = sources * nk, per = (all + parts - 1) / parts, first = part * per;
    const int steps = all - first < per ? all - first : per;
    u32x4 ra[2][OpA::PER], rb[2][NB][OpB::PER];
    // piece p of a chunk's PIECES: A's first, then each matrix's
    struct Chunk {
      typename OpA::From a;
      typename OpB::From b[NB];
      int k0, left;
    };
    auto chunk_at = [&](int step) {
      const int at = first + step;
      const bool second = at >= nk;
      const int k0 = (second ? at - nk : at) * BK;
      const int left = step < steps ? K - k0 : 0;
      Chunk c;
      c.k0 = k0;
      c.left = left;
      c.a = OpA::from(second ? s1.a : s0.a, lda, k0, left);
#pragma unroll
      for (int i = 0; i < NB; ++i) c.b[i] = OpB::from(second ? s1.b[i] : s0.b[i], ldb, k0, left);
      return c;
    };
    auto load = [&](auto& a, auto& b, const Chunk& c, int p) {
      if (p < OpA::PER) {
        if constexpr (A_MAPPED) {
          if (p == 0) opa.load_mapped(a, tid, s0.a, lda, a_map, c.k0, c.left);
        } else {
          a[p] = opa.load(c.a, tid, p);
        }
      } else {
        const int i = (p - OpA::PER) / OpB::PER, j = (p - OpA::PER) % OpB::PER;
        b[i][j] = opb.load(c.b[i], tid, j);
      }
    };
    auto store = [&](const auto& a, const auto& b, int buf, int p) {
      uint8_t* at = smem + buf * BUF_BYTES;
      if (p < OpA::PER) {
        OpA::store(a[p], tid, p, at);
      } else {
        const int i = (p - OpA::PER) / OpB::PER, j = (p - OpA::PER) % OpB::PER;
        OpB::store(b[i][j], tid, j, at + OpA::BYTES + i * OpB::BYTES);
      }
    };
    f32x4 xf[2][FM], wf[2][NB][FN];
    auto read = [&](int set, int buf, int s) {
      const uint8_t* at = smem + buf * BUF_BYTES;
#pragma unroll
      for (int fm = 0; fm < FM; ++fm) xf[set][fm] = OpA::frag(at, lane, (wm * FM + fm) * 32, s);
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
          wf[set][b][fn] = OpB::frag(at + OpA::BYTES + b * OpB::BYTES, lane, (wn * FN + fn) * 32, s);
    };
    // Chunk st is multiplied from buffer st & 1, while chunk st + 1 is stored from register set
    // (st + 1) & 1 into the other buffer (whose last reads, of chunk st - 1, are behind that chunk's barrier)
    // and the loads of chunk st + 3 go into the registers that frees.  A wave issues in order, and a 16-byte
    // store takes its turn for about 80 clocks and a load for about 40: they go out one at a time, each behind
    // a product that takes the matrix pipe 64 clocks, and each step's fragments are read a step ahead.  The
    // chunk's barrier stands in front of its last step, whose fragments have been read: its products cover the
    // reading of the next chunk's first ones.
    // (The fences keep that order: left alone, the compiler moves the reads to their first use.  A wave
    // without rows walks a loop of its own: a condition around the products would make every one of them
    // wait for all LDS traffic in flight.)
    auto chunk = [&](auto multiply, auto& a, auto& b, int buf, int st) {
      const Chunk next = chunk_at(st + 3);
      if constexpr (decltype(multiply)::value) {
        constexpr int BEHIND = PRODUCTS / STEPS * (STEPS - 1);  // products in front of the barrier
        // (with too few products for both in front of it the loads go on behind it)
        constexpr bool BOTH = BEHIND >= 2 * PIECES;
        constexpr int EVERY = BOTH ? BEHIND / (2 * PIECES) : 1;
        static_assert(BOTH || (PIECES <= BEHIND && 2 * PIECES <= PRODUCTS), "a product per store and load");
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
          if (s + 1 < STEPS) {
            read((s + 1) & 1, buf, s0k + s + 1);
          } else {
            lds_barrier();
            read(0, buf ^ 1, s0k);
          }
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int m = 0; m < NB; ++m)
#pragma unroll
              for (int fn = 0; fn < FN; ++fn)
#pragma unroll
                for (int fm = 0; fm < FM; ++fm) {
                  __builtin_amdgcn_sched_barrier(0);
                  f32x16& sum = acc[CHAINS == 2 ? s / (STEPS / 2) : 0][m][fn][fm];
                  sum = __builtin_amdgcn_mfma_f32_32x32x2f32(wf[s & 1][m][fn][j], xf[s & 1][fm][j], sum, 0, 0, 0);
                  const int done = (((s * 4 + j) * NB + m) * FN + fn) * FM + fm;
                  if ((!BOTH || done < BEHIND) && done % EVERY == 0) {
                    const int o = done / EVERY;
                    if (o < PIECES)
                      store(a, b, buf ^ 1, o);
                    else if (o < 2 * PIECES)
                      load(a, b, next, o - PIECES);
                  }
                }
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
#pragma unroll
        for (int p = 0; p < PIECES; ++p) store(a, b, buf ^ 1, p);
#pragma unroll
        for (int p = 0; p < PIECES; ++p) load(a, b, next, p);
        lds_barrier();
      }
    };
    auto load_all = [&](auto& a, auto& b, int step) {
      const Chunk c = chunk_at(step);
#pragma unroll
      for (int p = 0; p < PIECES; ++p) load(a, b, c, p);
      __builtin_amdgcn_sched_barrier(0);  // oldest first, as in the loop
    };
    load_all(ra[0], rb[0], 0);
    load_all(ra[1], rb[1], 1);
#pragma unroll
    for (int p = 0; p < PIECES; ++p) store(ra[0], rb[0], 0, p);
    load_all(ra[0], rb[0], 2);
    lds_barrier();
    auto walk = [&](auto multiply) {
      if constexpr (decltype(multiply)::value) read(0, 0, s0k);
      int st = 0;
      for (; st + 1 < steps; st += 2) {
        chunk(multiply, ra[1], rb[1], 0, st);
        chunk(multiply, ra[0], rb[0], 1, st + 1);
      }
      if (st < steps) chunk(multiply, ra[1], rb[1], 0, st);
    };
    if (active)
      walk(std::integral_constant<bool, true>{});
    else
      walk(std::integral_constant<bool, false>{});
    if constexpr (GROUPS == 2) {
      // the second group's sums onto the first's, through the chunks' LDS (the barrier: each chunk's last step reads the
      // next one's first fragments, the last chunk's too)
      constexpr int REGS = NB * FN * FM * 16;
      static_assert(2 * WM * REGS * 64 * 4 <= SMEM_BYTES, "the second group's sums fit the chunks' buffers");
      float* at = reinterpret_cast<float*>(smem) + (wm * 2 + wn) * (REGS * 64) + lane;
      auto exchange = [&](auto store) {
#pragma unroll
        for (int m = 0; m < NB; ++m)
#pragma unroll
          for (int fn = 0; fn < FN; ++fn)
#pragma unroll
            for (int fm = 0; fm < FM; ++fm)
#pragma unroll
              for (int i = 0; i < 16; ++i) {
                float& v = at[(((m * FN + fn) * FM + fm) * 16 + i) * 64];
                if constexpr (decltype(store)::value)
                  v = acc[0][m][fn][fm][i];
                else
                  acc[0][m][fn][fm][i] += v;
              }
      };
      const bool second = s0k != 0;
      lds_barrier();
      if (second && active) exchange(std::integral_constant<bool, true>{});
      lds_barrier();
      if (!second && active) exchange(std::integral_constant<bool, false>{});
    }
#pragma unroll
    for (int m = 0; m < NB; ++m)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int fm = 0; fm < FM; ++fm)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            sums[m][fn][fm][i] = CHAINS == 2 ? acc[0][m][fn][fm][i] + acc[CHAINS - 1][m][fn][fm][i] : acc[0][m][fn][fm][i];
  }
  // whether the wave holds the tile's sums after run
  static __device__ __forceinline__ bool holds_sums(int wave) { return wave_group(wave) == 0; }
};
}  // namespace f32t

// C = A B_e (+ A2 B2_e), or with DUAL C = SiLU(A B0_e) * (A B1_e), the two products left in g_keep and
// u_keep where those are given.  A block per tile; BLAYOUT as for the bf16 kernels.  With several rows of blocks
// (single products) each takes a part of the sum over K, and C is [gridDim.y][rows][N].
template <bool DUAL, int FM, int FN, int BLAYOUT, int GROUPS, int WM = 2>
__global__ __launch_bounds__(f32t::threads(GROUPS, WM), 2 * GROUPS) void glu_gemm_f32_kernel(
    const float* __restrict__ A, const float* __restrict__ B0, const float* __restrict__ B1,
    const float* __restrict__ A2, float* __restrict__ C, float* __restrict__ g_keep,
    float* __restrict__ u_keep, int K, int N, Groups g, int n_tiles) {
  constexpr int NB = DUAL ? 2 : 1;
  constexpr bool KN = BLAYOUT == FS2MOE_W_IN_OUT;
  using W = f32t::Walk<NB, FM, FN, false, KN, false, GROUPS, true, WM>;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[W::SMEM_BYTES];
  int e, row0, row_end, nt;
  if (!locate_tile_by_xcd<W::BM, W::THREADS>(g, n_tiles, reinterpret_cast<int32_t*>(smem), e, row0, row_end, nt)) return;
  e = __builtin_amdgcn_readfirstlane(e);
  row0 = __builtin_amdgcn_readfirstlane(row0);
  row_end = __builtin_amdgcn_readfirstlane(row_end);
  const int n0 = nt * W::BN;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = W::wave_m(wave), wn = W::wave_n(wave), lr = lane & 31, lk = lane >> 5;

  f32x16 acc[NB][FN][FM];

  const size_t at = (size_t)e * K * N + (KN ? (size_t)n0 : (size_t)n0 * K);
  typename W::Source s0, s1;
  s0.a = A + (size_t)row0 * K;
  s0.b[0] = B0 + at;
  s1 = s0;
  if constexpr (DUAL) {
    s0.b[1] = B1 + at;
  } else if (A2 != nullptr) {
    s1.a = A2 + (size_t)row0 * K;
    s1.b[0] = B1 + at;
  }
  const int m_wave = row0 + wm * 32 * FM;
  W::run(acc, smem, s0, s1, !DUAL && A2 != nullptr ? 2 : 1, K, KN ? N : K, K, row_end - row0, N - n0,
         m_wave < row_end, nullptr, DUAL ? 0 : (int)blockIdx.y, DUAL ? 1 : (int)gridDim.y);
  if (!W::holds_sums(wave)) return;
  if constexpr (!DUAL) C += (size_t)blockIdx.y * g.dense_rows * N;

#pragma unroll
  for (int fm = 0; fm < FM; ++fm) {
    const int m = m_wave + fm * 32 + lr;
    if (m >= row_end) continue;
#pragma unroll
    for (int fn = 0; fn < FN; ++fn)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = n0 + (wn * FN + fn) * 32 + 8 * q + 4 * lk;
        if (n >= N) continue;
        const size_t to = (size_t)m * N + n;
        f32x4 v, u;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[j] = acc[0][fn][fm][4 * q + j];
          u[j] = acc[NB - 1][fn][fm][4 * q + j];
        }
        if constexpr (DUAL) {
          if (g_keep != nullptr) {
            *reinterpret_cast<f32x4*>(g_keep + to) = v;
            *reinterpret_cast<f32x4*>(u_keep + to) = u;
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = (v[j] / (1.0f + expf(-v[j]))) * u[j];
        }
        *reinterpret_cast<f32x4*>(C + to) = v;
      }
  }
}

// One weight gradient: dW_e = A_e^T B_e over the rows of an expert (slots: the experts), or over seg_rows rows each of
// one group (slots: segments, whose sums go to `partial` where there are several).
struct F32WgradJob {
  const float *A, *B;
  float *C, *partial;
  int M, N, m_tiles, n_tiles, segments, seg_rows, rows;
  int grouped, first;  // first: its first block
};
// Those of a step in one launch: each alone ends with a round of tiles that leaves CUs idle.  1000 tokens, top-2 of 8,
// D 512, F 1408: three launches and the router's 113 us, one 89.
struct F32WgradJobs {
  static constexpr int MAX = 8;
  F32WgradJob job[MAX];
  int n;
};

// MAPPED: A's rows are read through a_map.
template <bool MAPPED>
__global__ __launch_bounds__(f32t::threads(1), 2) void grouped_wgrad_f32_kernel(
    const F32WgradJobs jobs, const int32_t* __restrict__ a_map, Groups g) {
  using W = f32t::Walk<1, 1, 1, true, true, MAPPED, 1, false>;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[W::SMEM_BYTES];
  int at = 0;
  for (int i = 1; i < jobs.n; ++i)
    if ((int)blockIdx.x >= jobs.job[i].first) at = i;
  const F32WgradJob& job = jobs.job[at];
  const float *A = job.A, *B = job.B;
  const int M = job.M, N = job.N, per = job.m_tiles * job.n_tiles;
  int slot = ((int)blockIdx.x - job.first) / per;
  const int rem = (int)blockIdx.x - job.first - slot * per;
  const int mt = rem / job.n_tiles, nt = rem - mt * job.n_tiles;
  int off, cnt;
  if (!job.grouped) {
    off = slot * job.seg_rows;
    cnt = job.rows - off < job.seg_rows ? job.rows - off : job.seg_rows;
  } else {
    off = __builtin_amdgcn_readfirstlane(g.offsets[slot]);
    cnt = __builtin_amdgcn_readfirstlane(g.counts[slot]);
  }
  const int m0 = mt * W::BM, n0 = nt * W::BN;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = W::wave_m(wave), wn = W::wave_n(wave), lr = lane & 31, lk = lane >> 5;
  f32x16 acc[1][1][1];
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[0][0][0][i] = 0.f;
  typename W::Source s;
  s.a = (MAPPED ? A : A + (size_t)off * M) + m0;
  s.b[0] = B + (size_t)off * N + n0;
  const int m_wave = m0 + wm * 32;
  if (cnt > 0) W::run(acc, smem, s, s, 1, M, N, cnt, M - m0, N - n0, m_wave < M,
                     MAPPED ? a_map + off : nullptr);
  float* to = job.partial != nullptr ? job.partial : job.C;
  to += (size_t)slot * M * N;
  const int m = m_wave + lr;
  if (m >= M) return;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int n = n0 + wn * 32 + 8 * q + 4 * lk;
    if (n >= N) continue;
    const f32x16& a = acc[0][0][0];
    *reinterpret_cast<f32x4*>(to + (size_t)m * N + n) = f32x4{a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
  }
}

}  // namespace fs2moe
