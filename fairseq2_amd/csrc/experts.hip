// Grouped SwiGLU expert GEMMs on MFMA.
//
// Both GEMMs of an expert network run as "grouped" GEMMs over the expert-contiguous row buffer:
//   H = SiLU(X Wg) * (X Wu)   (DUAL: two weight tiles share one activation tile, gate fused)
//   Y = H Wd
// A block owns a BM x BN output tile of one expert.  The tile -> (expert, row range) map is
// derived on the device from counts/offsets, so nothing is read back to the host.
//
// MFMA operand roles are swapped with respect to the textbook: the weight fragment is the "A"
// operand (rows = output channels n) and the activation fragment the "B" operand (columns = rows
// m of X), which yields the transposed tile.  In the 32x32 accumulator layout a lane then holds
// four CONSECUTIVE output channels of one row m, so results leave as 8-byte (bf16) or 16-byte
// (f32) stores without a trip through LDS.
//
// Expert weights are stored "in x out" (k-major rows, n contiguous: experts.py:53-82), but an MFMA
// operand lane needs 8 consecutive k for one n.  The tile is written to LDS as it lies in memory
// and read back with ds_read_tr16_b64, the gfx950 transposing LDS load: within 16 lanes, lane i
// receives element (i % 4) of lanes i/4, i/4 + 4, i/4 + 8, i/4 + 12 -- a 4(k) x 16(n) block
// transposed on the fly.  nn.Linear-oriented weights (the shared expert) are already k-contiguous
// and use plain 16-byte LDS reads.
#include "common.h"
#include "tile_map.h"
#include "experts_dma.h"
#include "experts_half.h"
#include "experts_f32.h"
#include "experts_fp8.h"
#include "experts_gemv.h"

namespace fs2moe {

// ------------------------------------------------------------------ bf16, 128-row tiles (64-bit addresses)
// For activation matrices of 4 GB and more, which the throughput kernel's 32-bit offsets do not reach.
namespace bf16k {
constexpr int BM = 128, BN = 128, BK = 64;
constexpr int LDA = BK + 8;    // sA row stride (elements): 144 B, conflict-free 16-byte reads
constexpr int LDB_KN = BN + 32;  // sB row stride for k-major tiles: 320 B
constexpr int LDB_NK = BK + 8;
}  // namespace bf16k

template <bool DUAL, int BLAYOUT>
__global__ __launch_bounds__(256, 2) void glu_gemm_bf16_kernel(
    const uint16_t* __restrict__ A, int lda, const uint16_t* __restrict__ B0,
    const uint16_t* __restrict__ B1, uint16_t* __restrict__ C, int ldc, int Kdim, int N, Groups g,
    int n_tiles) {
  using namespace bf16k;
  constexpr int NB = DUAL ? 2 : 1;
  constexpr bool KN = BLAYOUT == FS2MOE_W_IN_OUT;
  constexpr int SB_ELEMS = KN ? BK * LDB_KN : BN * LDB_NK;
  __shared__ __attribute__((aligned(16))) uint16_t sA[BM * LDA];
  __shared__ __attribute__((aligned(16))) uint16_t sB[NB][SB_ELEMS];

  const int tid = threadIdx.x;
  const int mt = blockIdx.x / n_tiles, nt = blockIdx.x - mt * n_tiles;
  int e, row0, row_end;
  if (!locate_tile<BM>(g, mt, e, row0, row_end)) return;
  const int n0 = nt * BN;
  const size_t wstride = (size_t)Kdim * N;
  const uint16_t* Bp[2] = {B0 + (size_t)e * wstride, DUAL ? B1 + (size_t)e * wstride : nullptr};

  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int lr = lane & 31, lk = lane >> 5;
  bool fm_active[2];
#pragma unroll
  for (int fm = 0; fm < 2; ++fm) fm_active[fm] = row0 + wm * 64 + fm * 32 < row_end;

  f32x16 acc[NB][2][2];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int fn = 0; fn < 2; ++fn)
#pragma unroll
      for (int fm = 0; fm < 2; ++fm)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[b][fn][fm][i] = 0.f;

  u32x4 ra[4], rb[NB][4];
  const u32x4 zero4 = {0u, 0u, 0u, 0u};

  auto load_global = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = tid + 256 * i;
      const int row = c >> 3, kc = c & 7;
      int grow = row0 + row;
      grow = grow < row_end ? grow : row_end - 1;
      const int k = k0 + kc * 8;
      ra[i] = k < Kdim ? *reinterpret_cast<const u32x4*>(A + (size_t)grow * lda + k) : zero4;
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = tid + 256 * i;
        if (KN) {
          const int k = k0 + (c >> 4), n = n0 + (c & 15) * 8;
          rb[b][i] = (k < Kdim && n < N)
                         ? *reinterpret_cast<const u32x4*>(Bp[b] + (size_t)k * N + n)
                         : zero4;
        } else {
          const int n = n0 + (c >> 3), k = k0 + (c & 7) * 8;
          rb[b][i] = (k < Kdim && n < N)
                         ? *reinterpret_cast<const u32x4*>(Bp[b] + (size_t)n * Kdim + k)
                         : zero4;
        }
      }
    }
  };
  auto store_lds = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = tid + 256 * i;
      *reinterpret_cast<u32x4*>(&sA[(c >> 3) * LDA + (c & 7) * 8]) = ra[i];
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = tid + 256 * i;
        if (KN)
          *reinterpret_cast<u32x4*>(&sB[b][(c >> 4) * LDB_KN + (c & 15) * 8]) = rb[b][i];
        else
          *reinterpret_cast<u32x4*>(&sB[b][(c >> 3) * LDB_NK + (c & 7) * 8]) = rb[b][i];
      }
    }
  };

  const int nk = (Kdim + BK - 1) / BK;
  load_global(0);
  for (int kt = 0; kt < nk; ++kt) {
    store_lds();
    __syncthreads();
    if (kt + 1 < nk) load_global((kt + 1) * BK);
    if (fm_active[0]) {
#pragma unroll
      for (int ks = 0; ks < BK / 16; ++ks) {
        bf16x8 xf[2];
#pragma unroll
        for (int fm = 0; fm < 2; ++fm)
          xf[fm] = lds_read_frag(&sA[(wm * 64 + fm * 32 + lr) * LDA + ks * 16 + lk * 8]);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
#pragma unroll
          for (int fn = 0; fn < 2; ++fn) {
            bf16x8 wf;
            if (KN) {
              const int s = lane & 15, half = (lane >> 4) & 1;
              const int kr = ks * 16 + lk * 8 + (s >> 2);
              const int col = wn * 64 + fn * 32 + half * 16 + (s & 3) * 4;
              wf = lds_read_frag_tr(&sB[b][kr * LDB_KN + col], &sB[b][(kr + 4) * LDB_KN + col]);
            } else {
              wf = lds_read_frag(&sB[b][(wn * 64 + fn * 32 + lr) * LDB_NK + ks * 16 + lk * 8]);
            }
            acc[b][fn][0] =
                __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf, xf[0], acc[b][fn][0], 0, 0, 0);
            if (fm_active[1])
              acc[b][fn][1] =
                  __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf, xf[1], acc[b][fn][1], 0, 0, 0);
          }
        }
      }
    }
    __syncthreads();
  }

  // Epilogue: lane holds, for row m, channels n = nb + 8q + 4*lk + {0..3}, q = 0..3.
#pragma unroll
  for (int fm = 0; fm < 2; ++fm) {
    const int m = row0 + wm * 64 + fm * 32 + lr;
    if (m >= row_end) continue;
#pragma unroll
    for (int fn = 0; fn < 2; ++fn) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = n0 + wn * 64 + fn * 32 + 8 * q + 4 * lk;
        if (n >= N) continue;
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (DUAL)
            v[j] = silu_f32(acc[0][fn][fm][4 * q + j]) * acc[NB - 1][fn][fm][4 * q + j];
          else
            v[j] = acc[0][fn][fm][4 * q + j];
        }
        u32x2 o = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        *reinterpret_cast<u32x2*>(C + (size_t)m * ldc + n) = o;
      }
    }
  }
}

// ------------------------------------------------------------------------------------ host
// One launch of the f32 kernel; a2, g_keep, u_keep may be null.
template <bool DUAL, int BLAYOUT>
static int launch_f32(const void* a, const void* b0, const void* b1, const void* a2, void* c,
                      void* g_keep, void* u_keep, int K, int N, const Groups& g, int64_t rows_bound,
                      const char* what, hipStream_t stream, int parts = 1) {
  const int groups = g.counts ? g.E : 0;
  const bool small = !f32t::large_tiles(DUAL, g.rows_to_plan(rows_bound), groups, N, 256);
  const bool flat = small && f32t::flat_tiles(DUAL, g.rows_to_plan(rows_bound), groups, N, parts, 256);
  const int bm = flat ? 32 : small ? 64 : 128, bn = small || DUAL ? 64 : 128;
  const int64_t m_tiles = rows_bound / bm + groups + 1;
  const int nt = (N + bn - 1) / bn;
  if (m_tiles * nt > 0x7ffffff0ll) {
    set_error("%s: grid too large", what);
    return FS2MOE_ERR_UNSUPPORTED;
  }
  // (small tiles of one product and flat ones: two groups of waves, f32t::threads)
  constexpr int groups_small = DUAL ? 1 : 2;
  auto k = flat    ? glu_gemm_f32_kernel<DUAL, 1, 1, BLAYOUT, 2, 1>
           : small ? glu_gemm_f32_kernel<DUAL, 1, 1, BLAYOUT, groups_small>
                   : glu_gemm_f32_kernel<DUAL, 2, DUAL ? 1 : 2, BLAYOUT, 1>;
  hipLaunchKernelGGL(k, dim3((unsigned)((m_tiles * nt + 7) / 8 * 8), (unsigned)parts),
                     dim3(flat ? f32t::threads(2, 1) : f32t::threads(small ? groups_small : 1)), 0, stream,
                     static_cast<const float*>(a), static_cast<const float*>(b0),
                     static_cast<const float*>(b1), static_cast<const float*>(a2),
                     static_cast<float*>(c), static_cast<float*>(g_keep), static_cast<float*>(u_keep), K,
                     N, g, nt);
  return check_launch(what);
}

// e4m3 weights go to the throughput kernels from this many rows per expert on (mean over all experts).  us of the layer,
// streamed against there, loaded evenly and by a popularity law of exponent 1.2:
//                                          20 rows             25                  28                  37
//   D 1024, F 1408, top-4 of 60      77, 98    68, 78    84, 99    76, 83    92, 99    80, 85   120, 101   93, 94
//   2048, 768, 8 of 128             166, 186  134, 146  178, 187  151, 157  188, 187  162, 159  236, 191  198, 172
//   4096, 6400, 2 of 16             273, 296  311, 310  305, 299  326, 337  325, 300  342, 353  432, 312  398, 372
//   4096, 1152, 8 of 32             123, 144  135, 146  130, 145  145, 147  145, 146  155, 148  193, 152  174, 155
//   3072, 1024, 6 of 64             158, 172  162, 192  174, 173  179, 198  183, 174  188, 198  244, 177  217, 203
//   2048, 12800, 2 of 8             163, 190  183, 213  179, 196  198, 217  200, 206  205, 220  247, 215  232, 230
//   5120, 2048, 1 of 16             133, 141  145, 153  152, 146  156, 165  156, 148  164, 173  201, 153  188, 192
//   1024, 4096, 2 of 16              70,  83   69,  91   78,  86   79,  96   84,  88   82,  97   104,  88   89,  97
// (from 25 on the large experts of an even load lose 1 to 6 % and all others gain up to 17; no size tells them apart
// from a skewed load, which the host does not see)
constexpr int64_t kFp8GemmMinRowsPerExpert = 27;
// Of a caller that does not say how many rows the experts have: so many of the buffers', which may have no padding.
constexpr int64_t kFp8GemmMinBufferRows = 32;

// The bf16 throughput kernel takes any D and F that are multiples of 8 (its KTAIL variants where a K is
// not a multiple of the unit's 64).  The entry points that exist for whole units only (the fused
// gather of the stage calls, the kept products, the two-source product) say so with this.
static bool whole_units(int act_dtype, int D, int F) {
  return act_dtype == FS2MOE_BF16 && D % (2 * dma::BK) == 0 && F % (2 * dma::BK) == 0;
}

// One launch of the bf16 kernel on smaller tiles (experts_half.h), one block per CU.
template <int BM, int BNV, bool DUAL, int BLAYOUT, bool KEEP_GU, bool TWO_SRC, bool ONCE>
static int launch_half_as(const void* a, const int32_t* row_map, int K, const void* b0, const void* b1,
                       const void* s0, const void* s1, void* c, int N, const Groups& g, const char* what,
                       int num_blocks, hipStream_t stream) {
  auto k = glu_gemm_half_kernel<BM, BNV, DUAL, BLAYOUT, KEEP_GU, TWO_SRC, ONCE>;
  constexpr int bytes = half_tiles::smem_bytes(BM, BNV, BLAYOUT), bn = DUAL ? BNV / 2 : BNV;
  static bool attr_set = false;  // benign race: setting the attribute is idempotent
  if (!attr_set) {
    hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) {
      set_error("%s: cannot reserve %d bytes of LDS: %s", what, bytes, hipGetErrorString(e));
      return FS2MOE_ERR_LAUNCH;
    }
    attr_set = true;
  }
  hipLaunchKernelGGL(k, dim3((unsigned)num_blocks), dim3(half_tiles::THREADS), bytes, stream,
                     static_cast<const uint8_t*>(a), row_map, K, static_cast<const uint8_t*>(b0),
                     static_cast<const uint8_t*>(b1), static_cast<const float*>(s0), static_cast<const float*>(s1),
                     static_cast<uint8_t*>(c), N, K, N, g, (N + bn - 1) / bn, HalfMx{});
  return check_launch(what);
}

template <int BM, int BNV, bool DUAL, int BLAYOUT, bool KEEP_GU, bool TWO_SRC>
static int launch_half(const void* a, const int32_t* row_map, int K, const void* b0, const void* b1,
                       const void* s0, const void* s1, void* c, int N, const Groups& g, const char* what,
                       int num_blocks, int64_t mean_rows, hipStream_t stream) {
  auto launch = g.once_past_cache && mean_rows <= half_tiles::once_rows(BM)
                    ? launch_half_as<BM, BNV, DUAL, BLAYOUT, KEEP_GU, TWO_SRC, true>
                    : launch_half_as<BM, BNV, DUAL, BLAYOUT, KEEP_GU, TWO_SRC, false>;
  return launch(a, row_map, K, b0, b1, s0, s1, c, N, g, what, num_blocks, stream);
}

// One launch of the bf16 throughput kernel on persistent blocks, one per CU (the 128 KB ring allows no
// more), a multiple of the 8 XCDs.  `b1`, `s0` and `s1` as the kernel's variants take them.
template <bool DUAL, int BLAYOUT, bool KEEP_GU = false, bool TWO_SRC = false>
static int launch_dma(const void* a, const int32_t* row_map, int K, const void* b0, const void* b1,
                      const void* s0, const void* s1, void* c, int N, Groups g,
                      int64_t rows_bound, const char* what, hipStream_t stream) {
  using namespace dma;
  constexpr bool CAN_TAIL = BLAYOUT != W_FP8_TILED;
  auto whole = glu_gemm_bf16_dma_kernel<DUAL, BLAYOUT, KEEP_GU, TWO_SRC>;
  auto tail = glu_gemm_bf16_dma_kernel<DUAL, BLAYOUT, KEEP_GU, TWO_SRC, CAN_TAIL>;
  auto whole_once = glu_gemm_bf16_dma_kernel<DUAL, BLAYOUT, KEEP_GU, TWO_SRC, false, false, true>;
  auto tail_once = glu_gemm_bf16_dma_kernel<DUAL, BLAYOUT, KEEP_GU, TWO_SRC, CAN_TAIL, false, true>;
  static bool attr_set = false;  // benign race: setting the attribute is idempotent
  if (!attr_set) {
    for (const void* k : {reinterpret_cast<const void*>(whole), reinterpret_cast<const void*>(tail),
                          reinterpret_cast<const void*>(whole_once), reinterpret_cast<const void*>(tail_once)}) {
      hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM_BYTES);
      if (e != hipSuccess) {
        set_error("%s: cannot reserve %d bytes of LDS: %s", what, SMEM_BYTES, hipGetErrorString(e));
        return FS2MOE_ERR_LAUNCH;
      }
    }
    attr_set = true;
  }
  const int num_blocks = cu_count_by_xcd();
  if (num_blocks == 0) {
    set_error("%s: cannot query the compute-unit count", what);
    return FS2MOE_ERR_LAUNCH;
  }
  const int groups = g.counts ? g.E : 0;
  // (rows that do not begin on lines share lines with the tiles beside: 16 experts of D 2048, F 3000, 512 tokens 174 us
  // without, 176 with)
  const bool on_lines = !CAN_TAIL || (BLAYOUT == FS2MOE_W_IN_OUT ? N : K) % 64 == 0;
  g.once_past_cache = on_lines && weights_past_cache(groups, pairs_of(g, rows_bound), K, N, CAN_TAIL ? 2 : 1);
  const int nt = (N + (DUAL ? 127 : 255)) / (DUAL ? 128 : 256);
  if ((rows_bound / BM + groups + 1) * nt > 0x7fffffffll) {
    set_error("%s: too many tiles", what);
    return FS2MOE_ERR_UNSUPPORTED;
  }
  const int64_t rows = pairs_of(g, rows_bound), mean_rows = groups ? rows / groups : rows;
  // (tiles of 64 x 64 are counted in 31 bits too)
  const bool counted = (rows_bound / 64 + groups + 1) * ((N + 63) / 64) <= 0x7fffffffll;
  constexpr bool SINGLE = !DUAL && CAN_TAIL;
  constexpr bool WHOLE_ROWS = DUAL && CAN_TAIL && !KEEP_GU && BLAYOUT == FS2MOE_W_IN_OUT;
  switch (counted ? half_tiles::pick(DUAL, CAN_TAIL, g.rows_to_plan(rows_bound), groups, K, N, num_blocks,
                                     WHOLE_ROWS ? g.most : 0)
                  : 0) {
    case 1:
      if constexpr (SINGLE)
        return launch_half<64, 64, DUAL, BLAYOUT, KEEP_GU, TWO_SRC>(a, row_map, K, b0, b1, s0, s1, c, N, g, what,
                                                                    num_blocks, mean_rows, stream);
      break;
    case 2:
      return launch_half<64, 128, DUAL, BLAYOUT, KEEP_GU, TWO_SRC>(a, row_map, K, b0, b1, s0, s1, c, N, g, what,
                                                                   num_blocks, mean_rows, stream);
    case 3:
      return launch_half<128, 128, DUAL, BLAYOUT, KEEP_GU, TWO_SRC>(a, row_map, K, b0, b1, s0, s1, c, N, g, what,
                                                                    num_blocks, mean_rows, stream);
    case 4:
      if constexpr (WHOLE_ROWS)
        return launch_half<64, 256, DUAL, BLAYOUT, KEEP_GU, TWO_SRC>(a, row_map, K, b0, b1, s0, s1, c, N, g, what,
                                                                     num_blocks, mean_rows, stream);
      break;
  }
  // The variant for any K also stores rows that do not begin on lines as L2 wants them, which counts for more than its
  // selects at every load where stores are a large part of the work: three results, or few units.  us with the variant
  // for whole units and with this one, 8 experts of 2000 rows, N 2728 and 60 of 300, N 712:
  //   K                            512        1024       1536       2048       3072       4096       5120
  //   three results (of 1500, pair) 165, 154  245, 240   354, 338   419, 398   595, 585   739, 725   913, 911
  //                                 82,  77   136, 130   187, 180   244, 240   349, 352   456, 459   564, 563
  //   gate/up (pair)               151, 149   249, 248   371, 372   468, 474   686, 696   916, 927  1133, 1154
  //                                 74,  73   127, 123   182, 175   234, 230   346, 345   455, 458   569, 572
  //   down's transpose              64,  60    98,  95   132, 128   168, 166   237, 239   317, 316   394, 393
  //                                 28,  29    45,  45    65,  62    81,  81   120, 124   155, 166   196, 205
  const bool off_lines =
      off_lines_variant(DUAL, BLAYOUT, TWO_SRC, CAN_TAIL) && N % 64 != 0 && (KEEP_GU || K <= 1536);
  // Weights past the caches where most tiles are their expert's only row block, by the mean of the experts' rows: a
  // choice for the launch, as in all kernels.  (By the expert, within the kernel, it costs more than it gives: two kinds
  // of loads into the same registers meet behind a branch, where the compiler waits for all of them.)  us without and with, experts loaded
  // evenly and by a popularity law of exponent 1.2; forward passes, then training steps with these rows on average:
  //   128 of D 2048, F 768    3  222, 204  102, 97    32  246, 227  181, 177    94  274, 257  259, 260
  //                         128  294, 283  319, 319  188  344, 336  393, 401   256  457, 475  456, 465
  //   8 of D 4096, F 8192   175  412, 431  467, 478
  //   128 of D 2048, F 768   64  908, 788  829, 776   128 1119, 980 1125, 1060  192 1321, 1227 1395, 1355
  //                         256 1535, 1586 1647, 1674
  //   64 of D 2048, F 1408  187  1170, 1116 1296, 1257  281 1531, 1607 1586, 1577
  const bool once =
      g.once_past_cache && mean_rows <= (KEEP_GU || BLAYOUT == FS2MOE_W_OUT_IN ? kOnceRowsTraining : kOnceRows);
  const bool units = K % (2 * BK) == 0 && !off_lines;
  hipLaunchKernelGGL(once ? (units ? whole_once : tail_once) : (units ? whole : tail), dim3((unsigned)num_blocks),
                     dim3(NWAVES * 64), SMEM_BYTES, stream, static_cast<const uint16_t*>(a), row_map, K,
                     static_cast<const uint16_t*>(b0), static_cast<const uint16_t*>(b1),
                     static_cast<const float*>(s0), static_cast<const float*>(s1),
                     static_cast<uint16_t*>(c), N, K, N, g, nt);
  return check_launch(what);
}

// Single products of few tiles over a long K: into how many parts the sum over K goes (1: it stays whole), each a
// round of tiles of its own.  The throughput kernel's time, in ns per unit of 64 k: a full round of heavy tiles 1950;
// a last one 1420 to 1820 with the CUs at work, a light tile counted as 0.6 of a heavy one; or, where it is dealt as
// halves, 1200 to 1400 with the light tiles (a whole launch of halves up to K 6000 1100), of light tiles alone 1000 to
// 1350; none faster than the operands come in (5 TB/s for both sources).  The smaller tiles' 300, 460 and 580 of one
// round.  Against that the parts' sums on their way out and in again, and a launch.  The figures are those that lose
// least over 229 products of 8 to 128 experts or one group, loaded evenly, at random or by a popularity law.  226 others
// take, whole, 1.094 times as long as by this rule, and 1.130 times as long as in the best number of parts; eleven are
// slower than whole by this rule, eight of them loaded by the law, which the host does not know.  us for two sources,
// whole (with the smaller tiles where they are taken) and in parts:
//   16 experts of 424 rows, K 13800, N 640    523, 360 (5)    8 of 427, K 9472, N 2112   439, 335 (3)
//   8 of 457, K 10560, N 512                  197, 104 (8)    8 of 880, K 8768, N 1216   427, 341 (3)
//   16 of 214, K 5568, N 1280                 181, 140 (3), with two 164
// and where it says 1: 16 of 552, K 7040, N 1088 355, 365 (3); 60 of 240, K 1600, N 1216 160, 192 (2); 16 of 375,
// K 1368, N 1024 46, 56 (2); 8 of 920, K 2800, N 576 88, 91 (2) and 87 (4).  A constant number of CUs, as the scratch is
// sized in calls that touch no device.
// f32 tiles (experts_f32.h): a CU multiplies no faster with several, so a part's time is its rounds of tiles, 0.53 us
// per 32 k and tile of 64 x 64.  8 experts of 250 rows, two sources of K 1408, N 512 (280 tiles): the step of 1000 tokens
// 394 -> 372 us in four parts, its loads at random (with 250 rows each the product is one round whole: 51 us, 53 in
// parts).  147 products, whole, 1.13 times as long as by this rule and 1.24 as in the best number of parts.
int split_parts(int sources, int64_t planned, int E, int K, int N, int dtype) {
  constexpr int CUS = 256, MIN_UNITS = 16;
  constexpr int64_t MAX_BYTES = 256ll << 20;
  const int groups = E > 0 ? E : 1;
  const int64_t real = planned - 15ll * E;  // (the experts' rows, equally loaded)
  if (real <= 0) return 1;
  // (the sums of buffers padded to 128 rows an expert have room in it)
  const int64_t part_bytes = (real + 127ll * E) * N * 4;
  if (dtype == FS2MOE_F32) {
    if (f32t::large_tiles(false, planned, E, N, CUS)) return 1;
    const int64_t each = real / groups, chunks = sources * ((K + f32t::BK - 1) / f32t::BK);
    // (half of a last row block per expert)
    const int64_t tiles = (groups + (each > 32 ? (real - 32 * groups) / 64 : 0)) * ((N + 63) / 64);
    auto time = [&](int64_t parts) { return (tiles * parts + CUS - 1) / CUS * ((chunks + parts - 1) / parts) * 530; };
    int best = 1;
    int64_t base = time(1);
    for (int parts = 2; parts <= 8 && chunks / parts >= MIN_UNITS && parts * part_bytes <= MAX_BYTES; ++parts) {
      const int64_t t = time(parts) + parts * planned * N / 500 + 6000;
      if (best == 1 ? t * 10 < base * 9 : t < base) {
        best = parts;
        base = t;
      }
    }
    const int64_t per = (chunks + best - 1) / best;
    return (int)((chunks + per - 1) / per);
  }
  const int64_t each = real / groups, nt = (N + dma::BNV - 1) / dma::BNV, rest = each % dma::BM;
  const int64_t heavy = (each / dma::BM + (rest > dma::LIGHT_ROWS)) * groups * nt;
  const int64_t light = (rest > 0 && rest <= dma::LIGHT_ROWS ? groups : 0) * nt;
  const int64_t units = (int64_t)sources * ((K + 63) / 64);
  const int64_t memory = sources * ((groups < real ? groups : real) * K * N + planned * K) / 2500;  // ns
  auto whole = [&](int64_t parts) {
    const int64_t left = heavy * parts % CUS, lights = light * parts, halves = 2 * left + lights;
    int64_t t = heavy * parts / CUS * 1950;  // of a unit
    if (halves > CUS) {
      const int64_t n = left + lights * 6 / 10;
      t += n / CUS * 1950 + (n % CUS ? 1420 + 400 * (n % CUS) / CUS : 0);
    } else if (left > 0) {
      t += (heavy < CUS && lights == 0 && parts == 1 && K < 6000 ? 1100 : 1200) + 200 * lights / CUS;
    } else if (lights > 0) {
      t += 1000 + 350 * lights / CUS;
    }
    t *= (units + parts - 1) / parts;
    return t > memory ? t : memory;
  };
  const int small = half_tiles::pick(false, true, planned, E, K, N, CUS);
  int64_t base = whole(1);
  if (small != 0) {
    const int64_t t = units * (small == 1 ? 300 : small == 2 ? 460 : 580);
    base = (t > memory ? t : memory) + 4000;
  }
  int best = 1;
  for (int parts = 2; parts <= 16 && units / parts >= MIN_UNITS && parts * part_bytes <= MAX_BYTES; ++parts) {
    const int64_t t = whole(parts) + parts * planned * N / 665 + 5000;
    // (worth 7.5 % by these figures, to be taken at all)
    if (best == 1 ? t * 40 < base * 37 : t < base) {
      best = parts;
      base = t;
    }
  }
  // (no part without a unit)
  const int64_t per = (units + best - 1) / best;
  return (int)((units + per - 1) / per);
}

// C [rows][N] = the sum of the parts [parts][rows][N] in order, rounded once, over the rows of group blockIdx.y (rows
// between the experts are left alone, there as here); a lane takes 8 columns of N, a multiple of 8.
template <typename T>
static __global__ __launch_bounds__(256) void split_sum_kernel(const float* __restrict__ from, int parts, int N,
                                                               Groups g, T* __restrict__ C) {
  const bool dense = g.counts == nullptr;
  const int64_t first = dense ? 0 : (int64_t)g.offsets[blockIdx.y] * N, all = (int64_t)g.dense_rows * N;
  const int64_t end = first + (int64_t)(dense ? g.dense_rows : g.counts[blockIdx.y]) * N;
  for (int64_t i = first + ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8; i < end; i += (int64_t)gridDim.x * 2048) {
    f32x4 lo = *reinterpret_cast<const f32x4*>(from + i), hi = *reinterpret_cast<const f32x4*>(from + i + 4);
#pragma unroll 4
    for (int p = 1; p < parts; ++p) {
      lo += *reinterpret_cast<const f32x4*>(from + (size_t)p * all + i);
      hi += *reinterpret_cast<const f32x4*>(from + (size_t)p * all + i + 4);
    }
    if constexpr (sizeof(T) == 2) {
      *reinterpret_cast<u32x4*>(C + i) = u32x4{pack_bf16x2(lo[0], lo[1]), pack_bf16x2(lo[2], lo[3]),
                                               pack_bf16x2(hi[0], hi[1]), pack_bf16x2(hi[2], hi[3])};
    } else {
      *reinterpret_cast<f32x4*>(C + i) = lo;
      *reinterpret_cast<f32x4*>(C + i + 4) = hi;
    }
  }
}
// (as many blocks a group as its planned rows have pieces of 2048, equally loaded)
template <typename T>
static int launch_split_sum(const void* scratch, int parts, int64_t planned, int N, const Groups& g, void* c,
                            hipStream_t stream) {
  const int64_t each = g.E * 2048ll, blocks = (planned * N + each - 1) / each;
  hipLaunchKernelGGL(split_sum_kernel<T>, dim3((unsigned)blocks, (unsigned)g.E), dim3(256), 0, stream,
                     static_cast<const float*>(scratch), parts, N, g, static_cast<T*>(c));
  return check_launch("split_sum");
}

// The product in `parts` parts (at least 2), whose sums go to scratch [parts][rows][N] f32, and their sum.
template <int BLAYOUT, bool TWO_SRC>
static int launch_split(const void* a, int K, const void* b0, const void* b1, const void* a2, void* c, int N,
                        const Groups& g, int64_t planned, int parts, void* scratch, const char* what, hipStream_t stream) {
  using namespace dma;
  auto k = glu_gemm_bf16_dma_kernel<false, BLAYOUT, false, TWO_SRC, true, true>;
  static bool attr_set = false;  // benign race: setting the attribute is idempotent
  if (!attr_set) {
    hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, SMEM_BYTES);
    if (e != hipSuccess) {
      set_error("%s: cannot reserve %d bytes of LDS: %s", what, SMEM_BYTES, hipGetErrorString(e));
      return FS2MOE_ERR_LAUNCH;
    }
    attr_set = true;
  }
  const int num_blocks = cu_count_by_xcd();
  if (num_blocks == 0) {
    set_error("%s: cannot query the compute-unit count", what);
    return FS2MOE_ERR_LAUNCH;
  }
  hipLaunchKernelGGL(k, dim3((unsigned)num_blocks), dim3(NWAVES * 64), SMEM_BYTES, stream,
                     static_cast<const uint16_t*>(a), static_cast<const int32_t*>(nullptr), K,
                     static_cast<const uint16_t*>(b0), static_cast<const uint16_t*>(b1),
                     static_cast<const float*>(a2), static_cast<const float*>(nullptr),
                     static_cast<uint16_t*>(scratch), parts, K, N, g, (N + 255) / 256 * parts);
  if (int rc = check_launch(what)) return rc;
  return launch_split_sum<uint16_t>(scratch, parts, planned, N, g, c, stream);
}

// The bf16 throughput kernel pair (gate/up, then down); BLAYOUT as the kernel takes it, scales only
// with dma::W_FP8_TILED.  With g_keep and u_keep the gate/up kernel also stores the two products (their
// destinations travel in the two scale arguments).
template <int BLAYOUT>
static int launch_dma_pair(const void* x, const int32_t* row_map, const Groups& g,
                           int64_t rows_bound, const void* w_gate, const void* w_up,
                           const void* w_down, const float* s_gate, const float* s_up,
                           const float* s_down, int D, int F, void* h, void* y,
                           hipStream_t stream, void* g_keep = nullptr, void* u_keep = nullptr) {
  constexpr bool CAN_KEEP = BLAYOUT != dma::W_FP8_TILED;
  if (g_keep != nullptr && !CAN_KEEP) {
    set_error("experts: the products are kept with bf16 weights only");
    return FS2MOE_ERR_UNSUPPORTED;
  }
  int rc;
  if (g_keep != nullptr)
    rc = launch_dma<true, BLAYOUT, CAN_KEEP>(x, row_map, D, w_gate, w_up, g_keep, u_keep, h, F, g,
                                             rows_bound, "glu_gemm_bf16_dma<gate,up>", stream);
  else
    rc = launch_dma<true, BLAYOUT>(x, row_map, D, w_gate, w_up, s_gate, s_up, h, F, g, rows_bound,
                                   "glu_gemm_bf16_dma<gate,up>", stream);
  if (rc) return rc;
  return launch_dma<false, BLAYOUT>(h, nullptr, F, w_down, nullptr, s_down, nullptr, y, D, g, rows_bound,
                                    "glu_gemm_bf16_dma<down>", stream);
}

// The throughput kernel addresses activations and one expert's weights with 32-bit byte offsets.
static bool dma_offsets_fit(int64_t rows_bound, int D, int F) {
  const int64_t wide = D > F ? D : F;
  return rows_bound * wide * 2 <= 0xffffffffll && (int64_t)D * F * 2 <= 0xffffffffll;
}

// The streaming pair for at most `rows_hint` rows per expert: see experts_gemv.h.  Measured on the
// Qwen3 layer shape (bf16 weights, whole layer, against the GEMM tiles): 1 token 44-47 against 69 us,
// 2 tokens 52 against 70, 3 tokens 56 against 71, 4 tokens 61 against 72; from 5 rows on the vector
// ALUs fall behind (8 tokens: 95 against 84 us), so the bound stops at 4 and the matrix-pipe stream
// below takes over.
#ifndef FS2MOE_GEMV_MAX_ROWS
#define FS2MOE_GEMV_MAX_ROWS 4
#endif
static bool gemv_applies(int act_dtype, int D, int F, const Groups& g, int rows_hint) {
  // (the stream kernels find their expert with four ballots over the counts: up to 256 experts)
  if (act_dtype != FS2MOE_BF16 || g.counts == nullptr || g.E > 256 || rows_hint < 1 ||
      rows_hint > FS2MOE_GEMV_MAX_ROWS)
    return false;
  const int r = rows_hint <= 1 ? 1 : rows_hint <= 2 ? 2 : 4;
  return gemv::offsets_fit(D, F) && gemv::fits(D > F ? D : F, r);
}

// How many experts' blocks are launched at a time, of about `blocks` in all.  More than run at once (two to
// a CU), since blocks that the hardware starts as others end balance better than blocks that go on to
// another expert (16 tokens, 81 experts: the down projection 60 us with 768, 57 with 2048); but a token or
// two reach a few experts only, and the blocks that find none take their time too (one token, the down
// projection: 7.2 us with 512 blocks, 10.6 with 2048).
static unsigned stream_experts(int blocks, int col_blocks, int E) {
  const int n = (blocks + col_blocks - 1) / col_blocks;
  return (unsigned)(n < E ? n : E);
}

// The shared expert's product that goes with the routed ones' gate/up or down product (shared null: none).
static DenseBeside dense_beside(const SharedBeside* shared, bool dual, const void* x, int D, const Selection* sel) {
  if (shared == nullptr || sel == nullptr) return DenseBeside{};
  auto in = [](const void* p) { return static_cast<const uint16_t*>(p); };
  if (dual)
    return {in(x), in(shared->gate), in(shared->up), static_cast<uint16_t*>(shared->h), D, shared->F, sel->T, (shared->F + 15) / 16};
  return {in(shared->h), in(shared->down), nullptr, static_cast<uint16_t*>(shared->out), shared->F, D, sel->T, (D + 15) / 16};
}
static unsigned beside_rows(const DenseBeside& dense, int col_blocks) {
  return (unsigned)((dense.blocks + col_blocks - 1) / col_blocks);
}
static size_t beside_lds(size_t bytes, const DenseBeside& dense, bool dual) {
  return dense.blocks > 0 && bytes < (size_t)dgemv::red_bytes(dual) ? (size_t)dgemv::red_bytes(dual) : bytes;
}

// A kernel that begins with the selection has a block a CU (its registers allow no more), which take (expert, channel block)
// pairs in turn, so that each selects once; and no more than there may be pairs (and blocks of the shared expert).
static dim3 selecting_grid(const Selection& sel, int col_blocks, int E, const DenseBeside& dense) {
  const int64_t pairs = (int64_t)sel.T * sel.K, most = (pairs < E ? pairs : E) * col_blocks + dense.blocks;
  return dim3((unsigned)(most < 256 ? most : 256));
}

template <int R, bool NT>
static int launch_gemv_pair_r(const void* x, const int32_t* row_map, const float* row_w,
                              const Groups& g, const void* w_gate, const void* w_up,
                              const void* w_down, int D, int F, void* h, void* y,
                              hipStream_t stream, const Selection* sel, const SharedBeside* shared) {
  using namespace gemv;
  auto k1 = glu_gemv_bf16_kernel<true, R, NT>;
  auto k1s2 = glu_gemv_bf16_kernel<true, R, NT, false, 2>;
  auto k1s4 = glu_gemv_bf16_kernel<true, R, NT, false, 4>;
  auto k2 = glu_gemv_bf16_kernel<false, R, NT>;
  auto k2d = glu_gemv_bf16_kernel<false, R, NT, true>;  // more loads in flight over a long K
  static bool attr_set = false;  // benign race: setting the attribute is idempotent
  if (!attr_set) {
    for (const void* k : {reinterpret_cast<const void*>(k1), reinterpret_cast<const void*>(k1s2),
                          reinterpret_cast<const void*>(k1s4), reinterpret_cast<const void*>(k2),
                          reinterpret_cast<const void*>(k2d)}) {
      const int bytes = k == reinterpret_cast<const void*>(k1s2) || k == reinterpret_cast<const void*>(k1s4)
                            ? MAX_LDS_SELECT : MAX_LDS_BYTES;
      if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
        set_error("experts: cannot reserve %d bytes of LDS", bytes);
        return FS2MOE_ERR_LAUNCH;
      }
    }
    attr_set = true;
  }
  if (sel != nullptr) k1 = g.E <= 128 ? k1s2 : k1s4;
  const Selection selection = sel != nullptr ? *sel : Selection{};
  const DenseBeside up_beside = dense_beside(shared, true, x, D, sel), down_beside = dense_beside(shared, false, x, D, sel);
  const uint16_t* xp = static_cast<const uint16_t*>(x);
  const int f_blocks = (F + COLS - 1) / COLS, d_blocks = (D + COLS - 1) / COLS;
  hipLaunchKernelGGL(k1, sel != nullptr ? selecting_grid(*sel, f_blocks, g.E, up_beside)
                                        : dim3((unsigned)f_blocks, stream_experts(256 * (R + 1), f_blocks, g.E)), dim3(threads(R)),
                     beside_lds((size_t)R * D * 2, up_beside, true), stream, xp, row_map, row_w, D, static_cast<const uint16_t*>(w_gate),
                     static_cast<const uint16_t*>(w_up), static_cast<uint16_t*>(h), F, D, F,
                     g.counts, g.offsets, g.E, selection, up_beside);
  if (int rc = check_launch("glu_gemv_bf16<gate,up>")) return rc;
  hipLaunchKernelGGL(deep_applies(F, R) ? k2d : k2,
                     dim3((unsigned)d_blocks, stream_experts(256 * (R + 1), d_blocks, g.E) + beside_rows(down_beside, d_blocks)),
                     dim3(threads(R)), beside_lds((size_t)R * F * 2, down_beside, false), stream, static_cast<const uint16_t*>(h),
                     static_cast<const int32_t*>(nullptr), static_cast<const float*>(nullptr), F,
                     static_cast<const uint16_t*>(w_down),
                     static_cast<const uint16_t*>(nullptr), static_cast<uint16_t*>(y), D, F, D,
                     g.counts, g.offsets, g.E, Selection{}, down_beside);
  return check_launch("glu_gemv_bf16<down>");
}

// The same for 5 to 16 rows per expert, on the matrix pipe (glu_gemv16_bf16_kernel).  Whole layer at
// the Qwen3 shape against the GEMM tiles: 5 tokens 57 against 72 us, 8 tokens 69-71 against 79, 12
// tokens 71 against 81, 16 tokens 78 against 83.  At 3 and 4 rows it ties with the vector-ALU stream (53.5
// against 52.4 and 56.5 against 57.6 us), at 1 and 2 it loses (48 against 41, 53 against 48: half as
// many blocks per expert).
#ifndef FS2MOE_GEMV16_MAX_ROWS
#define FS2MOE_GEMV16_MAX_ROWS 16
#endif
static bool gemv16_applies(int act_dtype, int D, int F, const Groups& g, int rows_hint) {
  if (act_dtype != FS2MOE_BF16 || g.counts == nullptr || g.E > 256 ||
      rows_hint <= FS2MOE_GEMV_MAX_ROWS || rows_hint > FS2MOE_GEMV16_MAX_ROWS)
    return false;
  return gemv::offsets_fit(D, F) && gemv16::fits(D > F ? D : F, 8);
}
// rows staged per pass: 16 when the bound asks for it and rows that long fit LDS, else 8 (an expert
// with more rows is walked again)
static int gemv16_rows(int D, int F, int rows_hint) {
  return rows_hint > 8 && gemv16::fits(D > F ? D : F, 16) ? 16 : 8;
}

template <int XR, bool NT>
static int launch_gemv16_pair(const void* x, const int32_t* row_map, const float* row_w,
                              const Groups& g, const void* w_gate, const void* w_up,
                              const void* w_down, int D, int F, void* h, void* y,
                              hipStream_t stream, const Selection* sel, const SharedBeside* shared) {
  using namespace gemv16;
  auto k1 = glu_gemv16_bf16_kernel<true, XR, NT>;
  auto k1s2 = glu_gemv16_bf16_kernel<true, XR, NT, 2>;
  auto k1s4 = glu_gemv16_bf16_kernel<true, XR, NT, 4>;
  auto k2 = glu_gemv16_bf16_kernel<false, XR, NT>;
  static bool attr_set = false;  // benign race: setting the attribute is idempotent
  if (!attr_set) {
    for (const void* k : {reinterpret_cast<const void*>(k1), reinterpret_cast<const void*>(k1s2),
                          reinterpret_cast<const void*>(k1s4), reinterpret_cast<const void*>(k2)}) {
      const int bytes = k == reinterpret_cast<const void*>(k1s2) || k == reinterpret_cast<const void*>(k1s4)
                            ? MAX_LDS_SELECT : MAX_LDS_BYTES;
      if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
        set_error("experts: cannot reserve %d bytes of LDS", bytes);
        return FS2MOE_ERR_LAUNCH;
      }
    }
    attr_set = true;
  }
  if (sel != nullptr) k1 = g.E <= 128 ? k1s2 : k1s4;
  const Selection selection = sel != nullptr ? *sel : Selection{};
  const DenseBeside up_beside = dense_beside(shared, true, x, D, sel), down_beside = dense_beside(shared, false, x, D, sel);
  const int f_blocks = (F + COLS - 1) / COLS, d_blocks = (D + COLS - 1) / COLS;
  hipLaunchKernelGGL(k1, sel != nullptr ? selecting_grid(*sel, f_blocks, g.E, up_beside)
                                        : dim3((unsigned)f_blocks, stream_experts(2048, f_blocks, g.E)), dim3(THREADS),
                     beside_lds(lds_bytes(D, XR, true), up_beside, true), stream, static_cast<const uint16_t*>(x), row_map, row_w, D,
                     static_cast<const uint16_t*>(w_gate), static_cast<const uint16_t*>(w_up),
                     static_cast<uint16_t*>(h), F, D, F, g.counts, g.offsets, g.E, selection, up_beside);
  if (int rc = check_launch("glu_gemv16_bf16<gate,up>")) return rc;
  hipLaunchKernelGGL(k2, dim3((unsigned)d_blocks, stream_experts(2048, d_blocks, g.E) + beside_rows(down_beside, d_blocks)),
                     dim3(THREADS), beside_lds(lds_bytes(F, XR, false), down_beside, false), stream, static_cast<const uint16_t*>(h),
                     static_cast<const int32_t*>(nullptr), static_cast<const float*>(nullptr), F,
                     static_cast<const uint16_t*>(w_down),
                     static_cast<const uint16_t*>(nullptr), static_cast<uint16_t*>(y), D, F, D,
                     g.counts, g.offsets, g.E, Selection{}, down_beside);
  return check_launch("glu_gemv16_bf16<down>");
}

// The dense SwiGLU (the shared expert, weights (N, K)) of up to 16 bf16 rows: dense_gemv_bf16_kernel.
// Llama-4 Scout's shared expert (D 5120, F 8192): 1 token 172 us on the GEMM tiles.
static bool dense_gemv_applies(int act_dtype, const Groups& g, int64_t rows) {
  return act_dtype == FS2MOE_BF16 && g.counts == nullptr && rows >= 1 && rows <= dgemv::MAX_ROWS;
}
template <bool NT>
static int launch_dense_gemv_pair(const void* x, int T, const void* w_gate, const void* w_up,
                                  const void* w_down, int D, int F, void* h, void* y,
                                  hipStream_t stream) {
  using namespace dgemv;
  hipLaunchKernelGGL((dense_gemv_bf16_kernel<true, NT>), dim3((unsigned)((F + 15) / 16)), dim3(THREADS), 0,
                     stream, static_cast<const uint16_t*>(x), D, static_cast<const uint16_t*>(w_gate),
                     static_cast<const uint16_t*>(w_up), static_cast<uint16_t*>(h), F, D, F, T);
  if (int rc = check_launch("dense_gemv_bf16<gate,up>")) return rc;
  hipLaunchKernelGGL((dense_gemv_bf16_kernel<false, NT>), dim3((unsigned)((D + 15) / 16)), dim3(THREADS), 0,
                     stream, static_cast<const uint16_t*>(h), F, static_cast<const uint16_t*>(w_down),
                     static_cast<const uint16_t*>(nullptr), static_cast<uint16_t*>(y), D, F, D, T);
  return check_launch("dense_gemv_bf16<down>");
}

// rows_hint: an upper bound on the rows of any one expert when the caller knows one (the number of
// tokens is one: a token takes an expert at most once), else 0.
template <int BLAYOUT>
static int launch_glu(const void* x, const int32_t* row_map, const Groups& g, int64_t rows_bound,
                      const void* w_gate, const void* w_up, const void* w_down, int D, int F,
                      int act_dtype, void* h, void* y, hipStream_t stream, int rows_hint = 0,
                      const float* row_w = nullptr, const Selection* sel = nullptr, const SharedBeside* shared = nullptr) {
  const int groups = g.counts ? g.E : 0;
  // (rows off the lines share them with the rows beside, in both orientations: nn.Linear's of D 4096, F 8192 42.8 us
  // without and 48.1 with the hint on the same weights again, 64.6 and 53.2 with other memory read in between; of D 5160,
  // F 8232 61.2, 99.4 and 96.4, 104.1; D 4104, F 8192 48.0, 61.1 and 68.8, 65.7; D 4096, F 8200 39.8, 51.7 and 63.8, 56.6,
  // one token each; 16 tokens 60, 80 and 84, 84; 49, 65 and 71, 69)
  const bool past = D % 64 == 0 && F % 64 == 0 && weights_past_cache(groups, pairs_of(g, rows_bound), D, F, 2);
  if constexpr (BLAYOUT == FS2MOE_W_OUT_IN) {
    if (row_map == nullptr && dense_gemv_applies(act_dtype, g, rows_bound)) {
      auto launch = past ? launch_dense_gemv_pair<true> : launch_dense_gemv_pair<false>;
      return launch(x, (int)rows_bound, w_gate, w_up, w_down, D, F, h, y, stream);
    }
  }
  if constexpr (BLAYOUT == FS2MOE_W_IN_OUT) {
    if (gemv_applies(act_dtype, D, F, g, rows_hint)) {
      auto launch = rows_hint <= 1   ? (past ? launch_gemv_pair_r<1, true> : launch_gemv_pair_r<1, false>)
                    : rows_hint <= 2 ? (past ? launch_gemv_pair_r<2, true> : launch_gemv_pair_r<2, false>)
                                     : (past ? launch_gemv_pair_r<4, true> : launch_gemv_pair_r<4, false>);
      return launch(x, row_map, row_w, g, w_gate, w_up, w_down, D, F, h, y, stream, sel, shared);
    }
    if (gemv16_applies(act_dtype, D, F, g, rows_hint)) {
      auto launch = gemv16_rows(D, F, rows_hint) == 8
                        ? (past ? launch_gemv16_pair<8, true> : launch_gemv16_pair<8, false>)
                        : (past ? launch_gemv16_pair<16, true> : launch_gemv16_pair<16, false>);
      return launch(x, row_map, row_w, g, w_gate, w_up, w_down, D, F, h, y, stream, sel, shared);
    }
  }
  if (row_w != nullptr || sel != nullptr) {
    set_error("experts: internal: row weights or a selection given to kernels that do not scale rows");
    return FS2MOE_ERR_UNSUPPORTED;
  }
  if (act_dtype == FS2MOE_BF16 && dma_offsets_fit(rows_bound, D, F))
    return launch_dma_pair<BLAYOUT>(x, row_map, g, rows_bound, w_gate, w_up, w_down, nullptr, nullptr,
                                    nullptr, D, F, h, y, stream);
  if (row_map != nullptr) {
    set_error("experts: the fused gather needs bf16 and activation matrices below 4 GB");
    return FS2MOE_ERR_UNSUPPORTED;
  }
  if (act_dtype == FS2MOE_BF16) {
    using namespace bf16k;
    const int64_t m_tiles = rows_bound / BM + groups + 1;
    const int nt1 = (F + BN - 1) / BN, nt2 = (D + BN - 1) / BN;
    if (m_tiles * nt1 > 0x7fffffffll || m_tiles * nt2 > 0x7fffffffll) {
      set_error("experts: grid too large");
      return FS2MOE_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL((glu_gemm_bf16_kernel<true, BLAYOUT>), dim3((unsigned)(m_tiles * nt1)),
                       dim3(256), 0, stream, static_cast<const uint16_t*>(x), D,
                       static_cast<const uint16_t*>(w_gate), static_cast<const uint16_t*>(w_up),
                       static_cast<uint16_t*>(h), F, D, F, g, nt1);
    if (int rc = check_launch("glu_gemm_bf16<gate,up>")) return rc;
    hipLaunchKernelGGL((glu_gemm_bf16_kernel<false, BLAYOUT>), dim3((unsigned)(m_tiles * nt2)),
                       dim3(256), 0, stream, static_cast<const uint16_t*>(h), F,
                       static_cast<const uint16_t*>(w_down), static_cast<const uint16_t*>(nullptr),
                       static_cast<uint16_t*>(y), D, F, D, g, nt2);
    return check_launch("glu_gemm_bf16<down>");
  }
  if (int rc = launch_f32<true, BLAYOUT>(x, w_gate, w_up, nullptr, h, nullptr, nullptr, D, F, g, rows_bound,
                                         "glu_gemm_f32<gate,up>", stream))
    return rc;
  return launch_f32<false, BLAYOUT>(h, w_down, nullptr, nullptr, y, nullptr, nullptr, F, D, g, rows_bound,
                                    "glu_gemm_f32<down>", stream);
}

}  // namespace fs2moe

using namespace fs2moe;

extern "C" int fs2moe_grouped_swiglu_fuses_gather(int32_t D, int32_t F, int32_t act_dtype,
                                                  int32_t w_dtype) {
  if (D <= 0 || F <= 0) return 0;
  if (w_dtype == FS2MOE_FP8_E4M3) return (act_dtype == FS2MOE_BF16 && D % 64 == 0 && F % 64 == 0) ? 1 : 0;
  return (w_dtype == act_dtype && whole_units(act_dtype, D, F)) ? 1 : 0;
}

extern "C" int fs2moe_grouped_swiglu_keeps(int32_t D, int32_t F, int64_t max_rows,
                                           int32_t act_dtype) {
  if (D <= 0 || F <= 0 || max_rows < 0) return 0;
  return (whole_units(act_dtype, D, F) && dma_offsets_fit(max_rows, D, F)) ? 1 : 0;
}

extern "C" int fs2moe_grouped_swiglu_keep(const void* xe, const int32_t* row_map,
                                          const int32_t* counts, const int32_t* offsets,
                                          const void* w_gate, const void* w_up, const void* w_down,
                                          int32_t E, int32_t D, int32_t F, int64_t max_rows,
                                          int32_t act_dtype, void* g, void* u, void* h, void* ye,
                                          void* stream) {
  FS2_REQUIRE(xe && counts && offsets && w_gate && w_up && w_down && g && u && h && ye,
              "grouped_swiglu_keep: null pointer");
  FS2_REQUIRE(E >= 1 && E <= FS2MOE_MAX_EXPERTS, "grouped_swiglu_keep: E=%d outside [1, %d]", E,
              FS2MOE_MAX_EXPERTS);
  FS2_REQUIRE(max_rows >= 0 && max_rows < (1ll << 31), "grouped_swiglu_keep: max_rows=%lld",
              (long long)max_rows);
  if (!fs2moe_grouped_swiglu_keeps(D, F, max_rows, act_dtype)) {
    set_error("grouped_swiglu_keep: needs bf16, D and F multiples of 64 and activation matrices "
              "below 4 GB (D=%d, F=%d, act_dtype %d, max_rows=%lld)",
              D, F, act_dtype, (long long)max_rows);
    return FS2MOE_ERR_UNSUPPORTED;
  }
  FS2_REQUIRE(aligned16(xe) && aligned16(w_gate) && aligned16(w_up) && aligned16(w_down) &&
                  aligned16(g) && aligned16(u) && aligned16(h) && aligned16(ye),
              "grouped_swiglu_keep: buffers must be 16-byte aligned");
  Groups grp{counts, offsets, E, 0};
  return launch_dma_pair<FS2MOE_W_IN_OUT>(xe, row_map, grp, max_rows, w_gate, w_up, w_down, nullptr,
                                          nullptr, nullptr, D, F, h, ye,
                                          static_cast<hipStream_t>(stream), g, u);
}

static int grouped_swiglu_impl(const void* xe, const int32_t* row_map, const int32_t* counts,
                               const int32_t* offsets, const void* w_gate, const void* w_up,
                               const void* w_down, const float* s_gate, const float* s_up,
                               const float* s_down, int32_t E, int32_t D, int32_t F,
                               int64_t max_rows, int64_t planned, int32_t act_dtype, int32_t w_dtype,
                               void* h, void* ye, int32_t rows_hint, void* stream,
                               const float* row_w = nullptr) {
  FS2_REQUIRE(xe && counts && offsets && w_gate && w_up && w_down && h && ye,
              "grouped_swiglu: null pointer");
  FS2_REQUIRE(row_w == nullptr || w_dtype == FS2MOE_BF16,
              "grouped_swiglu: internal: row weights go with bf16 weights");
  FS2_REQUIRE(rows_hint >= 0, "grouped_swiglu: rows_per_expert=%d", rows_hint);
  FS2_REQUIRE(E >= 1 && E <= FS2MOE_MAX_EXPERTS, "grouped_swiglu: E=%d outside [1, %d]", E,
              FS2MOE_MAX_EXPERTS);
  FS2_REQUIRE(D > 0 && F > 0 && D % 8 == 0 && F % 8 == 0,
              "grouped_swiglu: D=%d and F=%d must be positive multiples of 8", D, F);
  FS2_REQUIRE(max_rows >= 0 && max_rows < (1ll << 31), "grouped_swiglu: max_rows=%lld",
              (long long)max_rows);
  FS2_REQUIRE(act_dtype == FS2MOE_F32 || act_dtype == FS2MOE_BF16, "grouped_swiglu: act_dtype %d",
              act_dtype);
  FS2_REQUIRE(aligned16(xe) && aligned16(w_gate) && aligned16(w_up) && aligned16(w_down) &&
                  aligned16(h) && aligned16(ye),
              "grouped_swiglu: buffers must be 16-byte aligned");
  if (w_dtype == FS2MOE_FP8_E4M3) {
    // W8A16: e4m3 codes [E, F, D] / [E, D, F] with per-output-channel f32 scales.
    FS2_REQUIRE(act_dtype == FS2MOE_BF16, "grouped_swiglu: fp8 weights need bf16 activations");
    FS2_REQUIRE(s_gate && s_up && s_down, "grouped_swiglu: fp8 weights need scales");
    FS2_REQUIRE(D % 64 == 0 && F % 64 == 0,
                "grouped_swiglu: fp8 weights need D=%d and F=%d to be multiples of 64", D, F);
    FS2_REQUIRE(aligned16(s_gate) && aligned16(s_up) && aligned16(s_down),
                "grouped_swiglu: scales must be 16-byte aligned");
    if (max_rows == 0) return FS2MOE_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    // Two regimes.  With many rows per expert the layer is a GEMM: the bf16 throughput kernel, its
    // producers turning the codes into bf16 on the way to LDS (half the weight bytes of bf16, the
    // same matrix rate).  With few (decode) it is a stream over the weights: the kernels below.  The
    // row counts live on the device, so the choice goes by the mean number of rows per expert, whatever
    // the buffers are padded to; only where the caller does not say them by the buffers' rows.
    // (the streaming kernels build their item table with a thread per expert: up to 256 experts)
    Groups g{counts, offsets, E, 0, (int)planned};
    const int64_t pairs = pairs_of(g, max_rows);
    const bool many = g.planned > 0 ? pairs >= kFp8GemmMinRowsPerExpert * E : max_rows >= kFp8GemmMinBufferRows * E;
    if ((many || E > 256) && dma_offsets_fit(max_rows, D, F)) {
      return launch_dma_pair<dma::W_FP8_TILED>(xe, row_map, g, max_rows, w_gate, w_up, w_down, s_gate,
                                               s_up, s_down, D, F, h, ye, st);
    }
    FS2_REQUIRE(E <= 256, "grouped_swiglu: the e4m3 streaming kernels take up to 256 experts (E=%d)", E);
    // Persistent blocks, three to five per CU (what the kernels' registers allow), walking work
    // items.
    // A long K is split over the 4 waves of a block (the chain of dependent loads per wave sets the
    // time of an item), a short one over 2 with two sets of channel groups per block.  A wave takes
    // 2 (gate/up) or 4 (down) groups of 16 channels when K is long, half that when it is short;
    // N / 16 is a multiple of 4, so the channel blocks tile N exactly.  Figures with the kernel.
    // Chunks of 32 rows from 8 rows an expert on (6 rows: 1-4 % slower evenly, 3-8 % faster skewed; 9 and more:
    // 0-22 % faster); one group for gate/up up to 3 and 96 in all (16 experts 3-9 % faster, 128 1-8 %; more rows in
    // all, where those of the busy experts are read once more per group, by a popularity law: 60 tokens, top-8 of 256,
    // D 2048, F 1024 79 -> 89 us, 69, top-4 of 128, D 2496, F 1600 98 -> 102).  Of a caller that does not say the rows
    // neither, unless the buffers hold more than 8 rows an expert besides the padding to 16.
    const int cus = cu_count_by_xcd();
    if (cus == 0) {
      set_error("experts: cannot query the compute-unit count");
      return FS2MOE_ERR_LAUNCH;
    }
    // work items (chunks of at least 16 rows x channel blocks of at least 32 channels) are counted in 31 bits
    const int64_t chunks = max_rows / 16 + E;
    if (chunks * ((D > F ? D : F) / 32) > 0x7fffffffll) {
      set_error("experts: too many work items");
      return FS2MOE_ERR_UNSUPPORTED;
    }
    const bool fine_items = chunks * (F / 16) <= 0x7fffffffll;
    // (past the caches: chunks share an expert's weights in L2: 126 rows of 8 experts, D 1344, F 14080 140 us with them
    // there, 151 past it; 14 rows, D 4864, F 11136 260, 236; 64 tokens, top-8 of 128, D 2048, F 768 73.5, 70.4)
    const bool few = g.planned > 0 && pairs <= 3ll * E && pairs <= 96 && fine_items;
    auto launch = [&](auto dual_tag, auto fr_tag, auto nt_tag, const void* a, const int32_t* map, int lda,
                      const void* w0, const void* w1, const float* s0, const float* s1, void* c, int ldc, int kdim,
                      int n) {
      constexpr bool DUAL = decltype(dual_tag)::value, NT = decltype(nt_tag)::value;
      constexpr int FR = decltype(fr_tag)::value;
      auto go = [&](auto ks_tag, auto groups_tag) {
        constexpr int KS = decltype(ks_tag)::value, CGW = decltype(groups_tag)::value;
        const unsigned grid = (unsigned)(fp8w::blocks(DUAL, CGW, FR) * cus);
        hipLaunchKernelGGL((glu_gemm_fp8w_kernel<DUAL, KS, CGW, FR, NT>), dim3(grid), dim3(256), 0, st,
                           static_cast<const uint16_t*>(a), map, lda, static_cast<const uint8_t*>(w0),
                           static_cast<const uint8_t*>(w1), s0, s1, static_cast<uint16_t*>(c), ldc, kdim, n, counts,
                           offsets, E, n / (16 * CGW * (4 / KS)));
      };
      if (kdim < 512)
        return go(std::integral_constant<int, 2>{}, std::integral_constant<int, DUAL ? 1 : 2>{});
      if constexpr (DUAL && FR == 1)
        if (few) return go(std::integral_constant<int, 4>{}, std::integral_constant<int, 1>{});
      go(std::integral_constant<int, 4>{}, std::integral_constant<int, DUAL ? 2 : 4>{});
    };
    auto pair = [&](auto fr, auto nt) -> int {
      launch(std::true_type{}, fr, nt, xe, row_map, D, w_gate, w_up, s_gate, s_up, h, F, D, F);
      if (int rc = check_launch("glu_gemm_fp8w<gate,up>")) return rc;
      launch(std::false_type{}, fr, nt, h, nullptr, F, w_down, nullptr, s_down, nullptr, ye, D, F, D);
      return check_launch("glu_gemm_fp8w<down>");
    };
    if ((g.planned > 0 ? pairs : max_rows - 15ll * E) > 8ll * E)
      return pair(std::integral_constant<int, 2>{}, std::false_type{});
    if (g.planned > 0 && weights_past_cache(E, pairs, D, F, 1))
      return pair(std::integral_constant<int, 1>{}, std::true_type{});
    return pair(std::integral_constant<int, 1>{}, std::false_type{});
  }
  if (w_dtype != act_dtype) {
    set_error("grouped_swiglu: weight dtype %d with activation dtype %d has no kernel", w_dtype,
              act_dtype);
    return FS2MOE_ERR_UNSUPPORTED;
  }
  if (max_rows == 0) return FS2MOE_OK;
  Groups g{counts, offsets, E, 0, (int)planned};
  g.most = rows_hint;
  return launch_glu<FS2MOE_W_IN_OUT>(xe, row_map, g, max_rows, w_gate, w_up, w_down, D, F, act_dtype,
                                     h, ye, static_cast<hipStream_t>(stream), rows_hint, row_w);
}

bool fs2moe::swiglu_gathers_rows(int32_t act_dtype, int32_t w_dtype, int32_t D, int32_t F,
                                 int64_t max_rows) {
  if (act_dtype != FS2MOE_BF16 || D < 8 || F < 8 || D % 8 || F % 8) return false;
  if (w_dtype == FS2MOE_FP8_E4M3) return D % 64 == 0 && F % 64 == 0;
  return w_dtype == FS2MOE_BF16 && dma_offsets_fit(max_rows, D, F);
}

bool fs2moe::swiglu_streams_rows(int32_t act_dtype, int32_t w_dtype, int32_t D, int32_t F, int32_t E,
                                 int32_t rows_per_expert) {
  if (act_dtype != FS2MOE_BF16 || w_dtype != FS2MOE_BF16 || D < 8 || F < 8 || D % 8 || F % 8) return false;
  static const int32_t some = 0;  // (the predicates only ask whether the groups have counts)
  const Groups g{&some, &some, E, 0};
  return gemv_applies(act_dtype, D, F, g, rows_per_expert) || gemv16_applies(act_dtype, D, F, g, rows_per_expert);
}

bool fs2moe::swiglu_selects(int32_t act_dtype, int32_t w_dtype, int32_t D, int32_t F, int32_t E, int32_t T) {
  if (T < 1 || T > 16 || !swiglu_streams_rows(act_dtype, w_dtype, D, F, E, T)) return false;
  if (T <= FS2MOE_GEMV_MAX_ROWS) return (int64_t)D * (T <= 2 ? T : 4) * 2 <= gemv::MAX_LDS_SELECT;
  return gemv16::lds_bytes(D, gemv16_rows(D, F, T), true) <= (size_t)gemv16::MAX_LDS_SELECT;
}

int fs2moe::grouped_swiglu_selecting(const void* x, const Selection& sel, const void* w_gate, const void* w_up,
                                     const void* w_down, int32_t E, int32_t D, int32_t F, int64_t max_rows, int64_t planned,
                                     void* h, void* ye, const SharedBeside* shared, void* stream) {
  FS2_REQUIRE(swiglu_selects(FS2MOE_BF16, FS2MOE_BF16, D, F, E, sel.T),
              "grouped_swiglu: internal: D=%d F=%d E=%d of %d tokens do not select", D, F, E, sel.T);
  FS2_REQUIRE(aligned16(x) && aligned16(w_gate) && aligned16(w_up) && aligned16(w_down) && aligned16(h) && aligned16(ye),
              "grouped_swiglu: buffers must be 16-byte aligned");
  const Groups g{sel.counts, sel.offsets, E, 0, (int)planned};
  return launch_glu<FS2MOE_W_IN_OUT>(x, sel.perm, g, max_rows, w_gate, w_up, w_down, D, F, FS2MOE_BF16, h, ye,
                                     static_cast<hipStream_t>(stream), sel.T, sel.row_w, &sel, shared);
}

bool fs2moe::shared_goes_with_rows(int32_t D, int32_t F, int32_t T) {
  // (not where its weights are loaded past the caches, which these kernels choose for the routed ones)
  return T >= 1 && T <= dgemv::MAX_ROWS && D % 8 == 0 && F % 8 == 0 &&
         !(D % 64 == 0 && F % 64 == 0 && weights_past_cache(0, 0, D, F, 2));
}

int fs2moe::grouped_swiglu_scaled_rows(const void* x, const int32_t* row_map, const float* row_w,
                                       const int32_t* counts, const int32_t* offsets,
                                       const void* w_gate, const void* w_up, const void* w_down,
                                       int32_t E, int32_t D, int32_t F, int64_t max_rows, int64_t planned,
                                       void* h, void* ye, int32_t rows_per_expert, void* stream) {
  FS2_REQUIRE(row_map && row_w, "grouped_swiglu: null pointer");
  FS2_REQUIRE(swiglu_streams_rows(FS2MOE_BF16, FS2MOE_BF16, D, F, E, rows_per_expert),
              "grouped_swiglu: internal: D=%d F=%d E=%d with %d rows an expert do not stream", D, F, E,
              rows_per_expert);
  return grouped_swiglu_impl(x, row_map, counts, offsets, w_gate, w_up, w_down, nullptr, nullptr,
                             nullptr, E, D, F, max_rows, planned, FS2MOE_BF16, FS2MOE_BF16, h, ye,
                             rows_per_expert, stream, row_w);
}

extern "C" int fs2moe_grouped_swiglu(const void* xe, const int32_t* row_map, const int32_t* counts,
                                     const int32_t* offsets, const void* w_gate, const void* w_up,
                                     const void* w_down, const float* s_gate, const float* s_up,
                                     const float* s_down, int32_t E, int32_t D, int32_t F,
                                     int64_t max_rows, int32_t act_dtype, int32_t w_dtype, void* h,
                                     void* ye, void* stream) {
  return grouped_swiglu_impl(xe, row_map, counts, offsets, w_gate, w_up, w_down, s_gate, s_up, s_down,
                             E, D, F, max_rows, 0, act_dtype, w_dtype, h, ye, 0, stream);
}

extern "C" int fs2moe_grouped_swiglu_rows(const void* xe, const int32_t* row_map,
                                          const int32_t* counts, const int32_t* offsets,
                                          const void* w_gate, const void* w_up, const void* w_down,
                                          const float* s_gate, const float* s_up,
                                          const float* s_down, int32_t E, int32_t D, int32_t F,
                                          int64_t max_rows, int32_t act_dtype, int32_t w_dtype,
                                          void* h, void* ye, int32_t rows_per_expert, void* stream) {
  return grouped_swiglu_impl(xe, row_map, counts, offsets, w_gate, w_up, w_down, s_gate, s_up, s_down,
                             E, D, F, max_rows, 0, act_dtype, w_dtype, h, ye, rows_per_expert, stream);
}

extern "C" int fs2moe_grouped_swiglu_pairs(const void* xe, const int32_t* row_map,
                                           const int32_t* counts, const int32_t* offsets,
                                           const void* w_gate, const void* w_up, const void* w_down,
                                           const float* s_gate, const float* s_up,
                                           const float* s_down, int32_t E, int32_t D, int32_t F,
                                           int64_t max_rows, int32_t act_dtype, int32_t w_dtype,
                                           void* h, void* ye, int32_t rows_per_expert, int64_t pairs,
                                           void* stream) {
  FS2_REQUIRE(pairs >= 0 && pairs <= (max_rows > 0 ? max_rows : 0),
              "grouped_swiglu: %lld rows of experts in buffers of %lld", (long long)pairs, (long long)max_rows);
  return grouped_swiglu_impl(xe, row_map, counts, offsets, w_gate, w_up, w_down, s_gate, s_up, s_down, E, D, F,
                             max_rows, pairs > 0 ? planned_rows(pairs, E) : 0, act_dtype, w_dtype, h, ye,
                             rows_per_expert, stream);
}

int fs2moe::grouped_swiglu_planned(const void* xe, const int32_t* row_map, const int32_t* counts,
                                   const int32_t* offsets, const void* w_gate, const void* w_up, const void* w_down,
                                   const float* s_gate, const float* s_up, const float* s_down, int32_t E, int32_t D,
                                   int32_t F, int64_t max_rows, int64_t planned, int32_t act_dtype, int32_t w_dtype,
                                   void* h, void* ye, int32_t rows_per_expert, void* stream) {
  return grouped_swiglu_impl(xe, row_map, counts, offsets, w_gate, w_up, w_down, s_gate, s_up, s_down, E, D, F,
                             max_rows, planned, act_dtype, w_dtype, h, ye, rows_per_expert, stream);
}

// One grouped (or dense) GEMM, C = A @ B_e, on the kernels of the SwiGLU pair's second half.
template <int BLAYOUT>
static int launch_gemm(const void* a, const int32_t* row_map, const Groups& g, int64_t rows_bound,
                       const void* b, int K, int N, int dtype, void* c, hipStream_t stream) {
  const int groups = g.counts ? g.E : 0;
  if (dtype == FS2MOE_BF16 && dma_offsets_fit(rows_bound, K, N))
    return launch_dma<false, BLAYOUT>(a, row_map, K, b, nullptr, nullptr, nullptr, c, N, g, rows_bound,
                                      "glu_gemm_bf16_dma<single>", stream);
  if (row_map != nullptr) {
    set_error("gemm: a row map needs bf16 and matrices below 4 GB");
    return FS2MOE_ERR_UNSUPPORTED;
  }
  if (dtype == FS2MOE_BF16) {
    using namespace bf16k;
    const int64_t m_tiles = rows_bound / BM + groups + 1;
    const int nt = (N + BN - 1) / BN;
    if (m_tiles * nt > 0x7fffffffll) {
      set_error("gemm: grid too large");
      return FS2MOE_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL((glu_gemm_bf16_kernel<false, BLAYOUT>), dim3((unsigned)(m_tiles * nt)),
                       dim3(256), 0, stream, static_cast<const uint16_t*>(a), K,
                       static_cast<const uint16_t*>(b), static_cast<const uint16_t*>(nullptr),
                       static_cast<uint16_t*>(c), N, K, N, g, nt);
    return check_launch("glu_gemm_bf16<single>");
  }
  return launch_f32<false, BLAYOUT>(a, b, nullptr, nullptr, c, nullptr, nullptr, K, N, g, rows_bound,
                                    "glu_gemm_f32<single>", stream);
}

int fs2moe::grouped_gemm_planned(const void* a, const int32_t* row_map, const int32_t* counts, const int32_t* offsets,
                                 const void* b, int32_t b_layout, int32_t E, int32_t K, int32_t N, int64_t max_rows,
                                 int64_t planned, int32_t dtype, void* c, void* stream) {
  FS2_REQUIRE(a && b && c, "grouped_gemm: null pointer");
  FS2_REQUIRE((counts == nullptr) == (offsets == nullptr), "grouped_gemm: counts without offsets");
  FS2_REQUIRE(E >= 1 && E <= FS2MOE_MAX_EXPERTS && (counts != nullptr || E == 1),
              "grouped_gemm: E=%d", E);
  FS2_REQUIRE(b_layout == FS2MOE_W_IN_OUT || b_layout == FS2MOE_W_OUT_IN, "grouped_gemm: layout %d",
              b_layout);
  FS2_REQUIRE(dtype == FS2MOE_F32 || dtype == FS2MOE_BF16, "grouped_gemm: dtype %d", dtype);
  FS2_REQUIRE(K > 0 && N > 0 && K % 8 == 0 && N % 8 == 0,
              "grouped_gemm: K=%d and N=%d must be positive multiples of 8", K, N);
  FS2_REQUIRE(max_rows >= 0 && max_rows < (1ll << 31), "grouped_gemm: max_rows=%lld",
              (long long)max_rows);
  FS2_REQUIRE(aligned16(a) && aligned16(b) && aligned16(c),
              "grouped_gemm: buffers must be 16-byte aligned");
  if (max_rows == 0) return FS2MOE_OK;
  Groups g{counts, offsets, E, (int)max_rows, (int)planned};
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (b_layout == FS2MOE_W_IN_OUT)
    return launch_gemm<FS2MOE_W_IN_OUT>(a, row_map, g, max_rows, b, K, N, dtype, c, st);
  return launch_gemm<FS2MOE_W_OUT_IN>(a, row_map, g, max_rows, b, K, N, dtype, c, st);
}

extern "C" int fs2moe_grouped_gemm(const void* a, const int32_t* row_map, const int32_t* counts,
                                   const int32_t* offsets, const void* b, int32_t b_layout,
                                   int32_t E, int32_t K, int32_t N, int64_t max_rows, int32_t dtype,
                                   void* c, void* stream) {
  return grouped_gemm_planned(a, row_map, counts, offsets, b, b_layout, E, K, N, max_rows, 0, dtype, c, stream);
}

extern "C" int fs2moe_dense_swiglu_keep(const void* x, const void* w_gate, const void* w_up,
                                        const void* w_down, int32_t T, int32_t D, int32_t F,
                                        int32_t act_dtype, void* g, void* u, void* h, void* y,
                                        void* stream) {
  FS2_REQUIRE(x && w_gate && w_up && w_down && g && u && h && y, "dense_swiglu_keep: null pointer");
  FS2_REQUIRE(T >= 0, "dense_swiglu_keep: T=%d", T);
  if (!fs2moe_grouped_swiglu_keeps(D, F, T, act_dtype)) {
    set_error("dense_swiglu_keep: needs bf16, D and F multiples of 64 and activation matrices "
              "below 4 GB (D=%d, F=%d, act_dtype %d, T=%d)", D, F, act_dtype, T);
    return FS2MOE_ERR_UNSUPPORTED;
  }
  FS2_REQUIRE(aligned16(x) && aligned16(w_gate) && aligned16(w_up) && aligned16(w_down) &&
                  aligned16(g) && aligned16(u) && aligned16(h) && aligned16(y),
              "dense_swiglu_keep: buffers must be 16-byte aligned");
  if (T == 0) return FS2MOE_OK;
  Groups grp{nullptr, nullptr, 1, T};
  return launch_dma_pair<FS2MOE_W_OUT_IN>(x, nullptr, grp, T, w_gate, w_up, w_down, nullptr,
                                          nullptr, nullptr, D, F, h, y,
                                          static_cast<hipStream_t>(stream), g, u);
}

extern "C" int fs2moe_grouped_gemm_sum_supported(int32_t K, int32_t N, int64_t max_rows,
                                                 int32_t dtype) {
  if (K <= 0 || N <= 0 || max_rows < 0 || N % 8 != 0) return 0;
  return (dtype == FS2MOE_BF16 && K % (2 * dma::BK) == 0 && dma_offsets_fit(max_rows, K, N)) ? 1 : 0;
}

extern "C" int fs2moe_grouped_gemm_sum(const void* a1, const void* b1, const void* a2,
                                       const void* b2, const int32_t* counts,
                                       const int32_t* offsets, int32_t E, int32_t K, int32_t N,
                                       int64_t max_rows, int32_t dtype, void* c, void* stream) {
  FS2_REQUIRE(a1 && b1 && a2 && b2 && c, "grouped_gemm_sum: null pointer");
  FS2_REQUIRE((counts == nullptr) == (offsets == nullptr),
              "grouped_gemm_sum: counts without offsets");
  FS2_REQUIRE(E >= 1 && E <= FS2MOE_MAX_EXPERTS && (counts != nullptr || E == 1),
              "grouped_gemm_sum: E=%d", E);
  FS2_REQUIRE(max_rows >= 0 && max_rows < (1ll << 31), "grouped_gemm_sum: max_rows=%lld",
              (long long)max_rows);
  if (!fs2moe_grouped_gemm_sum_supported(K, N, max_rows, dtype)) {
    set_error("grouped_gemm_sum: needs bf16, K a multiple of 64, N a multiple of 8 and matrices "
              "below 4 GB (K=%d, N=%d, dtype %d, max_rows=%lld)",
              K, N, dtype, (long long)max_rows);
    return FS2MOE_ERR_UNSUPPORTED;
  }
  FS2_REQUIRE(aligned16(a1) && aligned16(b1) && aligned16(a2) && aligned16(b2) && aligned16(c),
              "grouped_gemm_sum: buffers must be 16-byte aligned");
  if (max_rows == 0) return FS2MOE_OK;
  // (the second activation matrix travels in the first scale argument, the second weights in B1)
  return launch_dma<false, FS2MOE_W_OUT_IN, false, true>(
      a1, nullptr, K, b1, b2, a2, nullptr, c, N, Groups{counts, offsets, E, (int)max_rows}, max_rows,
      "glu_gemm_bf16_dma<two sources>", static_cast<hipStream_t>(stream));
}

bool fs2moe::swiglu_train_applies(int32_t dtype, int32_t D, int32_t F, int64_t rows) {
  return dtype == FS2MOE_F32 || dma_offsets_fit(rows, D, F);
}

int fs2moe::swiglu_train(const void* x, const int32_t* row_map, const int32_t* counts,
                         const int32_t* offsets, int32_t E,
                         const void* w_gate, const void* w_up, const void* w_down, int32_t D,
                         int32_t F, int64_t rows, int64_t planned, int32_t dtype, void* g, void* u, void* h,
                         void* y, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  const Groups grp{E > 0 ? counts : nullptr, E > 0 ? offsets : nullptr, E > 0 ? E : 1, (int)rows, (int)planned};
  if (dtype == FS2MOE_BF16) {
    if (E > 0)
      return launch_dma_pair<FS2MOE_W_IN_OUT>(x, row_map, grp, rows, w_gate, w_up, w_down, nullptr, nullptr,
                                              nullptr, D, F, h, y, st, g, u);
    return launch_dma_pair<FS2MOE_W_OUT_IN>(x, nullptr, grp, rows, w_gate, w_up, w_down, nullptr, nullptr,
                                            nullptr, D, F, h, y, st, g, u);
  }
  int rc = E > 0 ? launch_f32<true, FS2MOE_W_IN_OUT>(x, w_gate, w_up, nullptr, h, g, u, D, F, grp, rows,
                                                     "glu_gemm_f32<gate,up>", st)
                 : launch_f32<true, FS2MOE_W_OUT_IN>(x, w_gate, w_up, nullptr, h, g, u, D, F, grp, rows,
                                                     "glu_gemm_f32<gate,up>", st);
  if (rc) return rc;
  return E > 0 ? launch_f32<false, FS2MOE_W_IN_OUT>(h, w_down, nullptr, nullptr, y, nullptr, nullptr, F, D,
                                                    grp, rows, "glu_gemm_f32<down>", st)
               : launch_f32<false, FS2MOE_W_OUT_IN>(h, w_down, nullptr, nullptr, y, nullptr, nullptr, F, D,
                                                    grp, rows, "glu_gemm_f32<down>", st);
}

int fs2moe::gemm_sum(const void* a1, const void* b1, const void* a2, const void* b2, int32_t layout,
                     const int32_t* counts, const int32_t* offsets, int32_t E, int32_t K, int32_t N,
                     int64_t rows, int64_t planned, int32_t dtype, void* c, void* split_scratch, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  const Groups g{E > 0 ? counts : nullptr, E > 0 ? offsets : nullptr, E > 0 ? E : 1, (int)rows, (int)planned};
  const int parts = split_parts(2, planned, E, K, N, dtype);
  if (parts > 1 && dtype == FS2MOE_F32) {
    const int rc = layout == FS2MOE_W_IN_OUT
                       ? launch_f32<false, FS2MOE_W_IN_OUT>(a1, b1, b2, a2, split_scratch, nullptr, nullptr, K, N, g,
                                                            rows, "glu_gemm_f32<two sources, parts>", st, parts)
                       : launch_f32<false, FS2MOE_W_OUT_IN>(a1, b1, b2, a2, split_scratch, nullptr, nullptr, K, N, g,
                                                            rows, "glu_gemm_f32<two sources, parts>", st, parts);
    return rc ? rc : launch_split_sum<float>(split_scratch, parts, planned, N, g, c, st);
  }
  if (parts > 1)
    return layout == FS2MOE_W_IN_OUT
               ? launch_split<FS2MOE_W_IN_OUT, true>(a1, K, b1, b2, a2, c, N, g, planned, parts, split_scratch,
                                                     "glu_gemm_bf16_dma<two sources, parts>", st)
               : launch_split<FS2MOE_W_OUT_IN, true>(a1, K, b1, b2, a2, c, N, g, planned, parts, split_scratch,
                                                     "glu_gemm_bf16_dma<two sources, parts>", st);
  // (the second activation matrix travels in the first scale argument, the second weights in B1)
  if (dtype == FS2MOE_BF16)
    return layout == FS2MOE_W_IN_OUT
               ? launch_dma<false, FS2MOE_W_IN_OUT, false, true>(a1, nullptr, K, b1, b2, a2, nullptr, c, N, g,
                                                                 rows, "glu_gemm_bf16_dma<two sources>", st)
               : launch_dma<false, FS2MOE_W_OUT_IN, false, true>(a1, nullptr, K, b1, b2, a2, nullptr, c, N, g,
                                                                 rows, "glu_gemm_bf16_dma<two sources>", st);
  return layout == FS2MOE_W_IN_OUT
             ? launch_f32<false, FS2MOE_W_IN_OUT>(a1, b1, b2, a2, c, nullptr, nullptr, K, N, g, rows,
                                                  "glu_gemm_f32<two sources>", st)
             : launch_f32<false, FS2MOE_W_OUT_IN>(a1, b1, b2, a2, c, nullptr, nullptr, K, N, g, rows,
                                                  "glu_gemm_f32<two sources>", st);
}

extern "C" int fs2moe_dense_swiglu(const void* x, const void* w_gate, const void* w_up,
                                   const void* w_down, int32_t T, int32_t D, int32_t F,
                                   int32_t act_dtype, void* h, void* y, void* stream) {
  FS2_REQUIRE(x && w_gate && w_up && w_down && h && y, "dense_swiglu: null pointer");
  FS2_REQUIRE(T >= 0 && D > 0 && F > 0 && D % 8 == 0 && F % 8 == 0,
              "dense_swiglu: T=%d, D=%d, F=%d (D and F must be positive multiples of 8)", T, D, F);
  FS2_REQUIRE(act_dtype == FS2MOE_F32 || act_dtype == FS2MOE_BF16, "dense_swiglu: act_dtype %d",
              act_dtype);
  FS2_REQUIRE(aligned16(x) && aligned16(w_gate) && aligned16(w_up) && aligned16(w_down) &&
                  aligned16(h) && aligned16(y),
              "dense_swiglu: buffers must be 16-byte aligned");
  if (T == 0) return FS2MOE_OK;
  Groups g{nullptr, nullptr, 1, T};
  return launch_glu<FS2MOE_W_OUT_IN>(x, nullptr, g, T, w_gate, w_up, w_down, D, F, act_dtype, h, y,
                                     static_cast<hipStream_t>(stream));
}
