// Shared device/host helpers for the gfx950 MoE kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fs2moe.h"

namespace fs2moe {

constexpr int kWave = 64;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(8))) short s16x8;
typedef __attribute__((ext_vector_type(2))) int i32x2;
typedef __attribute__((ext_vector_type(4))) int i32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;

// ---- memory that is read once -------------------------------------------------------------------
// Loads of what no other block reads and this one not again can carry the non-temporal hint: the line is the first that
// L2 gives up, the last-level cache does not take it, and memory delivers more.  Reads alone, 200 MB by 256 blocks:
// 6.1 TB/s without, 6.5 with; expert matrices by 256-byte pieces of their rows 5.8 and 6.4.
constexpr int kNonTemporal = 2;  // in a buffer instruction's cache policy
__device__ __forceinline__ u32x4 load_once(const void* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}
template <bool NT>
__device__ __forceinline__ u32x4 load_weights(const void* p) {
  if constexpr (NT) return load_once(p);
  return *reinterpret_cast<const u32x4*>(p);
}

// ---- bf16 <-> f32 (round to nearest even, NaN kept quiet) -------------------------------------
__device__ __forceinline__ float bf16_bits_to_f32(uint16_t b) {
  return __uint_as_float(((uint32_t)b) << 16);
}
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x0040u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
// Two floats -> packed bf16 pair in one v_cvt_pk_bf16_f32 (round to nearest even; lo in bits 0..15).
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  typedef __attribute__((ext_vector_type(2))) float f32x2_t;
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
  const f32x2_t v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}
// Two bf16 values times an f32 weight, each product rounded to bf16: what dispatch stores when it
// copies a row scaled by its routing weight, and what a kernel that scales the row on the way in
// must compute to give the same bits.
__device__ __forceinline__ uint32_t scale_bf16x2(uint32_t v, float w) {
  return pack_bf16x2(__uint_as_float(v << 16) * w, __uint_as_float(v & 0xffff0000u) * w);
}

template <typename T>
struct Elem;
template <>
struct Elem<float> {
  static __device__ __forceinline__ float load(const float* p) { return *p; }
  static __device__ __forceinline__ void store(float* p, float v) { *p = v; }
};
template <>
struct Elem<uint16_t> {  // bf16 bit pattern
  static __device__ __forceinline__ float load(const uint16_t* p) { return bf16_bits_to_f32(*p); }
  static __device__ __forceinline__ void store(uint16_t* p, float v) { *p = f32_to_bf16_bits(v); }
};

// v * sigmoid(v) with the hardware reciprocal (1 ulp), not a full-precision division.
__device__ __forceinline__ float silu_f32(float v) {
  return v * __builtin_amdgcn_rcpf(1.0f + __expf(-v));
}

// ---- wave-level helpers -------------------------------------------------------------------------
__device__ __forceinline__ int lane_id() { return threadIdx.x & (kWave - 1); }

// Wave-wide reductions on the DPP data path (no LDS round trips).  Four butterfly steps inside each
// row of 16 lanes (xor 1, xor 2, half-row mirror, row mirror), then row_bcast:15 into rows 1 and 3
// and row_bcast:31 into rows 2 and 3 leave the result in row 3; lane 63 is broadcast to all lanes.
constexpr int kDppXor1 = 0xB1;        // quad_perm:[1,0,3,2]
constexpr int kDppXor2 = 0x4E;        // quad_perm:[2,3,0,1]
constexpr int kDppHalfMirror = 0x141; // row_half_mirror
constexpr int kDppMirror = 0x140;     // row_mirror
constexpr int kDppBcast15 = 0x142;    // row_bcast:15
constexpr int kDppBcast31 = 0x143;    // row_bcast:31

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint64_t dpp_max_step_u64(uint64_t v) {
  const int lo = (int)(uint32_t)v, hi = (int)(uint32_t)(v >> 32);
  // lanes outside ROW_MASK (or without a source lane) keep their own value
  const uint32_t olo = (uint32_t)__builtin_amdgcn_update_dpp(lo, lo, CTRL, ROW_MASK, 0xf, false);
  const uint32_t ohi = (uint32_t)__builtin_amdgcn_update_dpp(hi, hi, CTRL, ROW_MASK, 0xf, false);
  const uint64_t o = ((uint64_t)ohi << 32) | olo;
  return o > v ? o : v;
}
__device__ __forceinline__ uint64_t wave_max_u64(uint64_t v) {
  v = dpp_max_step_u64<kDppXor1, 0xf>(v);
  v = dpp_max_step_u64<kDppXor2, 0xf>(v);
  v = dpp_max_step_u64<kDppHalfMirror, 0xf>(v);
  v = dpp_max_step_u64<kDppMirror, 0xf>(v);
  v = dpp_max_step_u64<kDppBcast15, 0xa>(v);
  v = dpp_max_step_u64<kDppBcast31, 0xc>(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, 63);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), 63);
  return ((uint64_t)hi << 32) | lo;
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_max_step_u32(uint32_t v) {
  // lanes outside ROW_MASK (or without a source lane) keep their own value
  const uint32_t o =
      (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, ROW_MASK, 0xf, false);
  return o > v ? o : v;
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  v = dpp_max_step_u32<kDppXor1, 0xf>(v);
  v = dpp_max_step_u32<kDppXor2, 0xf>(v);
  v = dpp_max_step_u32<kDppHalfMirror, 0xf>(v);
  v = dpp_max_step_u32<kDppMirror, 0xf>(v);
  v = dpp_max_step_u32<kDppBcast15, 0xa>(v);
  v = dpp_max_step_u32<kDppBcast31, 0xc>(v);
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_add_step_f32(float v) {
  // lanes outside ROW_MASK (or without a source lane) add zero
  const int o = __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xf, false);
  return v + __int_as_float(o);
}
__device__ __forceinline__ float wave_sum_f32(float v) {
  v = dpp_add_step_f32<kDppXor1, 0xf>(v);
  v = dpp_add_step_f32<kDppXor2, 0xf>(v);
  v = dpp_add_step_f32<kDppHalfMirror, 0xf>(v);
  v = dpp_add_step_f32<kDppMirror, 0xf>(v);
  v = dpp_add_step_f32<kDppBcast15, 0xa>(v);
  v = dpp_add_step_f32<kDppBcast31, 0xc>(v);
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ int dpp_add_step_i32(int v) {
  return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROW_MASK, 0xf, false);
}
__device__ __forceinline__ int wave_sum_i32(int v) {
  v = dpp_add_step_i32<kDppXor1, 0xf>(v);
  v = dpp_add_step_i32<kDppXor2, 0xf>(v);
  v = dpp_add_step_i32<kDppHalfMirror, 0xf>(v);
  v = dpp_add_step_i32<kDppMirror, 0xf>(v);
  v = dpp_add_step_i32<kDppBcast15, 0xa>(v);
  v = dpp_add_step_i32<kDppBcast31, 0xc>(v);
  return __builtin_amdgcn_readlane(v, 63);
}

// ---- MFMA operand fragments from LDS ---------------------------------------------------------------
// Plain: the lane's 8 consecutive k values lie contiguously (k-contiguous tile).
// Transposing: the tile is n-contiguous; ds_read_tr16_b64 hands lane i of each 16-lane group element
// (i % 4) of lanes i/4, i/4+4, i/4+8, i/4+12, i.e. a 4(k) x 16(n) block transposed.  p_lo / p_hi point at
// this lane's 4-element source chunk in k rows [k0, k0+4) and [k0+4, k0+8).
__device__ __forceinline__ bf16x8 lds_read_frag(const uint16_t* p) {
  return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(p));
}
__device__ __forceinline__ bf16x8 lds_read_frag_tr(const uint16_t* p_lo, const uint16_t* p_hi) {
  typedef __attribute__((address_space(3))) s16x4* lds_ptr;
  s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p_lo));
  s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p_hi));
  s16x8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  return __builtin_bit_cast(bf16x8, v);
}

// Block barrier that orders LDS traffic only.  __syncthreads() also fences global memory, for which
// the compiler drains every outstanding global load (s_waitcnt vmcnt(0)); loops that keep a register
// set of loads in flight across their barriers, and synchronise on nothing that lives in global
// memory, use this one.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// 8 e4m3 codes (two dwords) -> 8 bf16 values, all exact.  One instruction for two (two to f32 and one to join their upper
// halves before: 1000 tokens, top-2 of 8, D 2048, F 12800 463, 434 us; 150, top-8 of 32, D 4096, F 1152 172, 149).
__device__ __forceinline__ bf16x8 fp8x8_to_bf16x8(uint32_t lo, uint32_t hi) {
  u32x4 out;
  const int w[2] = {(int)lo, (int)hi};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    out[2 * i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[i], 1.f, false));
    out[2 * i + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[i], 1.f, true));
  }
  return __builtin_bit_cast(bf16x8, out);
}

// ---- host side -----------------------------------------------------------------------------------
void set_error(const char* fmt, ...);
int check_launch(const char* what);

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
// Compute units of the current device, rounded down to a multiple of its 8 XCDs (0 on failure).
inline int cu_count_by_xcd() {
  static int cached = 0;  // benign race: every thread computes the same value
  if (cached == 0) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus < 8)
      return 0;
    cached = cus / 8 * 8;
  }
  return cached;
}

inline int elem_size(int dtype) { return dtype == FS2MOE_F32 ? 4 : dtype == FS2MOE_BF16 ? 2 : 1; }

// What is left of router and dispatch where the experts' first kernel does it itself (swiglu_selects): the partial logits
// [slices][T][E], and where its results go.
struct Selection {
  const float *partial, *bias;
  int slices, T, K, score_fn, renormalize, tile_m;
  int64_t max_rows;
  int32_t* topk_idx;
  float* topk_w;
  int32_t *counts, *offsets, *perm, *inv_perm;
  float* row_w;
};

// Where the whole-layer call wants its dispatch (no rows copied): with at most 32 bf16 tokens the
// router's finishing kernel ends with it; with more the finishing kernel, or the block that routes a
// whole tile of 32 tokens from an (E, D) matrix, also counts its tile's pairs per expert and ranks them
// (up to kIndexTilesMax tiles), which leaves one dispatch kernel to run (dispatch_index_tiles); all set `done`.  At
// any other size the router leaves `done` false and the caller runs fs2moe_dispatch.  Either way the
// arrays hold the same values.  `ws` is the dispatch workspace (fs2moe_dispatch_workspace_bytes).
struct DispatchAfterRouter {
  int tile_m;
  int64_t max_rows;
  int32_t *counts, *offsets, *perm, *inv_perm;
  void* ws;
  int64_t ws_bytes;
  // optional (bf16 decode sizes, rows scaled by the routing weight on their way into the experts
  // instead of by a copy): per expert row the weight of its pair, written next to perm
  float* row_w;
  // optional: may take the selection instead (partial is set then) where the router leaves partial logits of at most
  // kRouterTileTok tokens and is not asked for logits; `done` is set as well
  Selection* later;
  bool done;
};
constexpr int kRouterTileTok = 32;   // tokens per tile of the MFMA routers
constexpr int kIndexTilesMax = 512;  // tiles whose counts every block of dispatch_index_tiles adds up
// The dispatch workspace as the tile-counting router fills it: per tile and expert the number of the
// tile's tokens that chose the expert (a byte: at most 32; E up to a multiple of 8 of them), then per
// pair its rank among the tile's pairs of the same expert.
inline uint8_t* tile_counts_of(void* ws) { return static_cast<uint8_t*>(ws); }
inline int32_t* tile_rank_of(void* ws, int T, int E, int tile_tok) {
  const int64_t nt = (T + tile_tok - 1) / tile_tok;
  return reinterpret_cast<int32_t*>(static_cast<uint8_t*>(ws) + (nt * ((E + 7) / 8 * 8) + 255) / 256 * 256);
}
// The rest of dispatch after such a router: offsets, counts, perm and inv_perm as fs2moe_dispatch
// writes them without a row copy, for tiles of tile_tok (8 or more, at most 32) tokens.  E at most 256; at
// most kIndexTilesMax tiles.
int dispatch_index_tiles(const int32_t* topk_idx, int32_t T, int32_t K, int32_t E, int tile_tok, int32_t tile_m,
                         int64_t max_rows, const uint8_t* tile_counts, const int32_t* tile_rank,
                         int32_t* counts, int32_t* offsets, int32_t* perm, int32_t* inv_perm,
                         void* stream);
// fs2moe_router_topk (xn null) or fs2moe_router_topk_norm; logits may be null
int router_then_dispatch(const void* x, const void* norm_w, float norm_eps, void* xn,
                         const void* router, const float* bias, int32_t T, int32_t D, int32_t E,
                         int32_t K, int32_t act_dtype, int32_t score_fn, int32_t renormalize,
                         int32_t* topk_idx, float* topk_w, float* logits, void* workspace, int64_t workspace_bytes,
                         DispatchAfterRouter* disp, void* stream);

// fs2moe_dispatch without a row copy that also writes row_w[row] = topk_w[pair] (see
// DispatchAfterRouter): at most 256 tokens and 256 experts, K <= 16 or not.
int dispatch_with_row_weights(const int32_t* topk_idx, const float* topk_w, int32_t T, int32_t K,
                              int32_t E, int32_t tile_m, int64_t max_rows, int32_t* counts,
                              int32_t* offsets, int32_t* perm, int32_t* inv_perm, float* row_w,
                              void* stream);
// The experts' rows that a plan goes by: as many as `pairs` rows take in blocks of 16, whatever granularity the buffers
// have.  Where the plan decides how sums are cut, results then do not depend on the padding.
inline int64_t planned_rows(int64_t pairs, int E) { return pairs + 15ll * E; }
// fs2moe_grouped_swiglu_rows, fs2moe_grouped_swiglu_w8a8 and fs2moe_grouped_gemm for callers that know the planned rows
// (most stage calls know the buffers' size alone, and plan by that).
int grouped_swiglu_planned(const void* xe, const int32_t* row_map, const int32_t* counts, const int32_t* offsets,
                           const void* w_gate, const void* w_up, const void* w_down, const float* s_gate,
                           const float* s_up, const float* s_down, int32_t E, int32_t D, int32_t F, int64_t max_rows,
                           int64_t planned, int32_t act_dtype, int32_t w_dtype, void* h, void* ye,
                           int32_t rows_per_expert, void* stream);
int grouped_swiglu_w8a8_planned(const void* xq, const void* xs, const int32_t* row_map, const int32_t* counts,
                                const int32_t* offsets, const void* w_gate, const void* w_up, const void* w_down,
                                const float* s_gate, const float* s_up, const float* s_down, int32_t E, int32_t D,
                                int32_t F, int64_t x_rows, int64_t max_rows, int64_t planned, void* hq, void* hs,
                                void* ye, void* stream);
int grouped_gemm_planned(const void* a, const int32_t* row_map, const int32_t* counts, const int32_t* offsets,
                         const void* b, int32_t b_layout, int32_t E, int32_t K, int32_t N, int64_t max_rows,
                         int64_t planned, int32_t dtype, void* c, void* stream);
// Whether the grouped SwiGLU pair of these sizes reads its rows through a row map (no gathered copy).
bool swiglu_gathers_rows(int32_t act_dtype, int32_t w_dtype, int32_t D, int32_t F, int64_t max_rows);
// Whether the grouped SwiGLU pair of these sizes runs on the kernels that stream the weights past a
// few staged rows (at most rows_per_expert of any expert), which can scale each row by row_w as
// they stage it; and that pair: fs2moe_grouped_swiglu_rows with rows read through row_map and
// multiplied by row_w[row] (rounded to bf16, as dispatch's scaled copy rounds them).
bool swiglu_streams_rows(int32_t act_dtype, int32_t w_dtype, int32_t D, int32_t F, int32_t E,
                         int32_t rows_per_expert);
// Whether the pair may begin with the selection itself (grouped_swiglu_selecting): up to 16 tokens on these kernels, with room
// for its tables in LDS; and that pair, whose rows are those of `sel`, read from x.
// (shared: optionally a shared expert, computed in the same launches)
struct SharedBeside {
  const void *gate, *up, *down;
  int F;
  void *h, *out;
};
bool swiglu_selects(int32_t act_dtype, int32_t w_dtype, int32_t D, int32_t F, int32_t E, int32_t T);
int grouped_swiglu_selecting(const void* x, const Selection& sel, const void* w_gate, const void* w_up, const void* w_down,
                             int32_t E, int32_t D, int32_t F, int64_t max_rows, int64_t planned, void* h, void* ye,
                             const SharedBeside* shared, void* stream);
// Whether a shared expert of F features can go with it, for at most 16 tokens.
bool shared_goes_with_rows(int32_t D, int32_t F, int32_t T);
int grouped_swiglu_scaled_rows(const void* x, const int32_t* row_map, const float* row_w,
                               const int32_t* counts, const int32_t* offsets, const void* w_gate,
                               const void* w_up, const void* w_down, int32_t E, int32_t D, int32_t F,
                               int64_t max_rows, int64_t planned, void* h, void* ye,
                               int32_t rows_per_expert, void* stream);

// ---- pieces of a training step (fs2moe_train_forward / fs2moe_train_backward)
// Whether the SwiGLU pair keeps its two products at these sizes, and that pair (E 0: one group of `rows`
// rows with nn.Linear-oriented weights; bf16: rows read through row_map where it is not null).
bool swiglu_train_applies(int32_t dtype, int32_t D, int32_t F, int64_t rows);
int swiglu_train(const void* x, const int32_t* row_map, const int32_t* counts, const int32_t* offsets, int32_t E,
                 const void* w_gate, const void* w_up, const void* w_down, int32_t D, int32_t F,
                 int64_t rows, int64_t planned, int32_t dtype, void* g, void* u, void* h, void* y, void* stream);
// Work beside the caller's stream: from fork() on what is given to stream() runs on a stream of the library's own, behind
// what the caller's had at mark() (or, without one, at fork()), and join() has the caller's wait for it, so that a caller sees one stream's worth of
// ordering (and a capturing stream captures both branches).  Where `wanted` is false, or there is no such stream to have without ordering callers' streams,
// stream() is the caller's and the other three do nothing: which it is, beside() says from the beginning, so that it decides
// where in the order of calls the branch's work stands.  A branch that is forked is joined on every way out.
class Branch {
 public:
  Branch(bool wanted, void* stream);
  Branch(const Branch&) = delete;
  Branch& operator=(const Branch&) = delete;
  ~Branch();
  bool beside() const { return side_ != nullptr; }
  void* stream() const;
  int mark();
  int fork();
  int join();

 private:
  struct SideStream* side_ = nullptr;
  void* main_;
  bool marked_ = false, forked_ = false;
};
// Whether more than 16 tokens' shared expert pays as a branch beside the routed experts.  What it gains is the ends of the
// other's launches, where CUs run out of tiles, and its small ones: 2 to 10 % of a call.  What it costs is the host's time
// for two pairs of record and wait, 30 us a pass and more after other work: a loss wherever the host is what a call waits
// for.  So by what the pass should take the GPU: the weights at 5 TB/s and the products at 60 % of the pipes' rate, 130 us of
// them forward, 200 backward, which multiplies twice.  us without and with the branch (which estimate):
//   forward 56, 90 (26: 137 tokens, D 576, F 576, top-4 of 32); 92, 101 (60); 100, 110 (75); 120, 129 (117: 1122, D 704, F
//   1408, top-4 of 60); 164, 172 (116); 177, 164 (132: 349 of f32, D 768, F 2048, 16); 181, 162 (185: 100, D 2048, F 4096,
//   16); 192, 179 (179); 280, 276 (253); 421, 394; 782, 747; 2734, 2627 (6000, D 5120, F 8192, 8)
//   training, backward pass 520, 508 (230: 3001 tokens, D 1024, F 1368, top-2 of 16); 526, 492 (252: 263 of f32, D 1024, F
//   2048, top-2 of 8); 409, 416 (185: 700, D 1024, F 4096, top-2 of 8, both passes; as a first pass 520, 590)
// late: a pass whose branch brings less or costs more, 350 us forward.  That is one behind a router that normalises the
// rows, whose branch begins with the experts' launches, which stream weights as fast alone where a call is mostly that:
//   199.6, 203.4 (191: 100 tokens, D 2048, F 4096, top-2 of 16); 205.6, 207.5 (211: 200); 249.6, 256.1 (322: 600, D 2048, F
//   1408, top-6 of 64); 372, 366 (395: 40, D 4096, F 8192, top-2 of 8); 375, 363 (453: 577 of f32, D 640, F 1728, top-6 of
//   64); 506, 491 (600: 1854, D 2496, F 4352, top-2 of 8); 475, 462 (549: 5000, D 1024, F 4096, top-2 of 8); 838, 819 (1194)
// and the forward pass of a training step, whose host time is not hidden in a first pass or where a program waits:
//   508, 496, but as a first pass 620, 665 (129: the 3001 tokens above); 775, 764 and 862, 903 (267: 1800, D 2048, F 2048,
//   top-2 of 16); 493, 489 and 617, 705 (152: 900, D 1536, F 3072, top-2 of 8); 495, 467 and 596, 621 (149: 263 of f32)
// Time with the branch over time without it in 70 drawn calls, queued behind others, then with the host waiting for each:
// where the rule says yes, forward 17 calls 0.96 (0.91 to 1.01), 0.97 (0.91 to 1.02), behind a router that normalises 6 0.96
// (0.91 to 0.99), 0.96; training steps 18 0.98 (0.93 to 1.03), 0.97 (0.92 to 1.02).  Where it says no and a branch was
// forced, in front of the router: 5 1.27, 1.08; 13 1.06, 1.02; 11 1.17, 1.09.
bool branch_pays(int T, int K, int E, int D, int F, int F_shared, int act_dtype, int w_dtype, bool late, bool backward);
// Into how many parts the sum over K of a product of `sources` pairs of matrices goes (1: it stays whole), by the
// planned rows (E 0: the rows).
int split_parts(int sources, int64_t planned, int E, int K, int N, int dtype);
// c = a1 @ B1 + a2 @ B2 (fs2moe_grouped_gemm's layouts and groups; E 0: one group), one rounding: in split_parts(2,
// planned, ..) parts, for whose sums there is scratch [parts][rows][N] f32.
int gemm_sum(const void* a1, const void* b1, const void* a2, const void* b2, int32_t layout,
             const int32_t* counts, const int32_t* offsets, int32_t E, int32_t K, int32_t N,
             int64_t rows, int64_t planned, int32_t dtype, void* c, void* split_scratch, void* stream);
// One of several weight gradients taken together: grouped (over the experts' rows) or over all `rows` of
// one group.
struct WgradRequest {
  const void *a, *b;
  void* dw;
  int32_t M, N;
  bool grouped;
  int segments;  // set by wgrad_plan: of a group's rows, each with its own partial sums
  bool map_a = false, map_b = false;  // bf16: the operand's rows are read through the row map
};
// Cuts the rows of single groups whose tiles would take longer than the others together (the experts' `planned`
// rows); returns the bytes of scratch that the partial sums need.
int64_t wgrad_plan(WgradRequest* r, int n, int32_t E, int64_t planned, int64_t rows, int32_t dtype);
int wgrad_all(const WgradRequest* r, int n, const int32_t* row_map, const int32_t* counts, const int32_t* offsets,
              int32_t E, int64_t grouped_rows, int64_t rows, int32_t dtype, void* scratch, void* stream);
// fs2moe_router_backward into rows of ld >= E elements, those past E zero
int router_backward_ld(const float* logits, const int32_t* topk_idx, const float* topk_w,
                       const float* d_w, int32_t T, int32_t E, int32_t K, int32_t score_fn,
                       int32_t renormalize, int32_t dtype, void* dlogits, int32_t ld, void* stream);

}  // namespace fs2moe

#define FS2_REQUIRE(cond, ...)          \
  do {                                  \
    if (!(cond)) {                      \
      fs2moe::set_error(__VA_ARGS__);   \
      return FS2MOE_ERR_ARG;            \
    }                                   \
  } while (0)
