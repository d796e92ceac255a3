// A training step of the whole layer: one call per pass over the stages of the other files.
//
// The host path matters here as much as the kernels: a step is 25 to 40 launches, and calling each from
// Python with its own buffers took the host longer (10 to 15 us a launch) than a layer of a few
// thousand rows takes the GPU.  Both calls therefore carve every intermediate out of two buffers and
// launch the whole pass.  What is new on the device is small: the gather of the output gradients, which
// also takes the dot products that are the combine weights' gradients, the activation's derivative of a
// step whose rows stay in token order, and the padding of a router matrix whose number of experts is not
// a multiple of 8.
#include <algorithm>

#include "common.h"

namespace fs2moe {

// One wave per (token, slot) pair p with row r = inv_perm[p]: dye[r] = dout[t] * w (w the pair's combine
// weight where it scales the output, else 1), and then d_w[p] = <ye[r], dout[t]> (ye is not read otherwise).
// A pair without a row (an expert id out of range) has a zero gradient.  Same products, sums and roundings as
// the row copy of fs2moe_dispatch and fs2moe_pair_dot, whose passes over dout and launches it replaces.  With
// weighted 0 it is a plain copy of rows, of x as well.
template <typename T>
__global__ __launch_bounds__(256) void gather_backward_kernel(
    const T* __restrict__ dout, const T* __restrict__ ye, const int32_t* __restrict__ inv_perm,
    const float* __restrict__ topk_w, int pairs, int K, int D, int weighted, T* __restrict__ dye,
    float* __restrict__ d_w) {
  const int p = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (p >= pairs) return;
  const int lane = threadIdx.x & 63;
  const int row = __builtin_amdgcn_readfirstlane(inv_perm[p]);
  if (row < 0) {
    if (d_w != nullptr && lane == 0) d_w[p] = 0.f;
    return;
  }
  constexpr int VEC = 16 / sizeof(T);
  const int chunks = D / VEC;
  const u32x4* src = reinterpret_cast<const u32x4*>(dout) + (size_t)(p / K) * chunks;
  const u32x4* yr = reinterpret_cast<const u32x4*>(ye) + (size_t)row * chunks;
  u32x4* dst = reinterpret_cast<u32x4*>(dye) + (size_t)row * chunks;
  const float w = weighted ? topk_w[p] : 1.f;
  float s = 0.f;
  for (int c = lane; c < chunks; c += 64) {
    const u32x4 g = src[c];
    u32x4 y = {0u, 0u, 0u, 0u};
    if (weighted) y = yr[c];
    u32x4 o = g;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (sizeof(T) == 2) {
        if (weighted) {
          o[j] = scale_bf16x2(g[j], w);
          s += __uint_as_float(y[j] << 16) * __uint_as_float(g[j] << 16);
          s += __uint_as_float(y[j] & 0xffff0000u) * __uint_as_float(g[j] & 0xffff0000u);
        }
      } else if (weighted) {
        o[j] = __float_as_uint(__uint_as_float(g[j]) * w);
        s += __uint_as_float(y[j]) * __uint_as_float(g[j]);
      }
    }
    dst[c] = o;
  }
  if (!weighted) return;
  s = wave_sum_f32(s);
  if (lane == 0) d_w[p] = s;
}

// The same for a step whose rows stay in token order (in_token_order below): one wave per pair p with row
// r = inv_perm[p].  dh holds the products of the token's output gradient, not yet weighted, with the expert's
// down projection; from the kept g and u come h (weighted: the left operand of that projection's gradient,
// whose right one is the unweighted output gradient), dg and du, and from the forward pass' h the combine
// weight's gradient d_w[p] = <ye[r], dout[t]> = <h[r], dh[r]>, which so needs neither ye nor dout.  (With an
// h from the rounded g and u the router's gradient is 15% further from 64 bits: three roundings instead of
// two.)  Bound by memory: seven passes over [rows, F].  h may be dh's buffer.  What the forward pass kept is read here for
// the last time, past the caches (load_once), which changes little: us of a training step without and with the hint, 260
// tokens, top-1 of 8, F 6400 243, 243; 2048, top-4 of 32, F 512 237, 237; 4096, top-8 of 128, F 768 1514, 1513; 8000,
// top-2 of 16, F 1024 357, 353; 700, top-2 of 8, F 8192 1350, 1357.
__global__ __launch_bounds__(256) void swiglu_backward_pairs_kernel(
    const uint16_t* __restrict__ g, const uint16_t* __restrict__ u, const uint16_t* __restrict__ h_fwd,
    const uint16_t* dh, const int32_t* __restrict__ inv_perm, const float* __restrict__ topk_w, int pairs, int F,
    uint16_t* h, uint16_t* __restrict__ dg, uint16_t* __restrict__ du, float* __restrict__ d_w) {
  const int p = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (p >= pairs) return;
  const int lane = threadIdx.x & 63;
  const int row = __builtin_amdgcn_readfirstlane(inv_perm[p]);
  if (row < 0) {
    if (lane == 0) d_w[p] = 0.f;
    return;
  }
  const float w = topk_w[p];
  const size_t base = (size_t)row * F;
  float dot = 0.f;
  for (int c = lane * 8; c < F; c += 512) {
    const u32x4 gv = load_once(g + base + c), uv = load_once(u + base + c), fv = load_once(h_fwd + base + c);
    const u32x4 dv = *reinterpret_cast<const u32x4*>(dh + base + c);
    u32x4 hv, gov, uov;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float ho[2], go[2], uo[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const float gf = __uint_as_float(q ? gv[j] & 0xffff0000u : gv[j] << 16);
        const float uf = __uint_as_float(q ? uv[j] & 0xffff0000u : uv[j] << 16);
        const float df = __uint_as_float(q ? dv[j] & 0xffff0000u : dv[j] << 16);
        const float s = 1.0f / (1.0f + __expf(-gf)), silu = gf * s, dw = df * w;
        dot += __uint_as_float(q ? fv[j] & 0xffff0000u : fv[j] << 16) * df;
        ho[q] = silu * uf * w;
        go[q] = dw * uf * (s * (1.0f + gf * (1.0f - s)));
        uo[q] = dw * silu;
      }
      hv[j] = pack_bf16x2(ho[0], ho[1]);
      gov[j] = pack_bf16x2(go[0], go[1]);
      uov[j] = pack_bf16x2(uo[0], uo[1]);
    }
    *reinterpret_cast<u32x4*>(h + base + c) = hv;
    *reinterpret_cast<u32x4*>(dg + base + c) = gov;
    *reinterpret_cast<u32x4*>(du + base + c) = uov;
  }
  dot = wave_sum_f32(dot);
  if (lane == 0) d_w[p] = dot;
}

// out[r, 0..cols_out) = in[r, 0..cols_in), cut or padded with zeros
template <typename T>
__global__ __launch_bounds__(256) void copy_columns_kernel(const T* __restrict__ in, int cols_in,
                                                           T* __restrict__ out, int cols_out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int64_t r = i / cols_out;
  const int c = (int)(i - r * cols_out);
  out[i] = c < cols_in ? in[r * cols_in + c] : (T)0;
}

static int copy_columns(const void* in, int cols_in, void* out, int cols_out, int64_t rows, int dtype,
                        hipStream_t st) {
  const int64_t n = rows * cols_out;
  const dim3 grid((unsigned)((n + 255) / 256)), block(256);
  if (dtype == FS2MOE_BF16)
    hipLaunchKernelGGL(copy_columns_kernel<uint16_t>, grid, block, 0, st, static_cast<const uint16_t*>(in),
                       cols_in, static_cast<uint16_t*>(out), cols_out, n);
  else
    hipLaunchKernelGGL(copy_columns_kernel<float>, grid, block, 0, st, static_cast<const float*>(in),
                       cols_in, static_cast<float*>(out), cols_out, n);
  return check_launch("copy_columns");
}

namespace {
struct Carver {
  uint8_t* base;
  int64_t used = 0;
  void* take(int64_t bytes) {
    void* p = base != nullptr ? base + used : nullptr;
    used += (bytes + 255) / 256 * 256;
    return p;
  }
};
using Args = fs2moe_train_args;

int64_t rows_of(const Args& a) { return FS2MOE_MAX_ROWS(a.T, a.K, a.E, a.tile_m); }
int64_t planned_rows(const Args& a) { return fs2moe::planned_rows((int64_t)a.T * a.K, a.E); }
int padded_experts(const Args& a) { return (a.E + 7) / 8 * 8; }
// With up to 16 bf16 tokens the experts run as streams over their weights, as in the inference call, and
// keep no products: the backward pass computes them again.
bool streams(const Args& a) {
  return a.T <= 16 && swiglu_streams_rows(a.act_dtype, a.act_dtype, a.D, a.F, a.E, a.T);
}

// Whether the rows stay in token order: the products read the tokens' rows (x, and in the backward pass dout)
// through the permutation, the weights on the output are applied to dh and h in f32
// (swiglu_backward_pairs_kernel), and nothing of K rows a token is kept.  Needs rows that enter the experts
// unscaled, and the bf16 kernels, which take a row map.
bool in_token_order(const Args& a) { return a.act_dtype == FS2MOE_BF16 && !a.scale_input && !streams(a); }
// Whether the weight gradients, too, read them there.  Copies in expert order (of x, of dout) are two passes;
// without them each tile of 256 columns of F gathers the rows anew, and a chunk of rows takes it longer, which
// the largest expert's tiles, chains of their chunks, pay in full.  So: in place up to four such tiles and up to
// 768 rows an expert on average, and with so few rows (under two chunks of 32) that a tile is mostly its results.
// Steps without copies against with them, us, experts equally loaded:
//   8192 tokens, D 2048, F 512 / 768 of 128, 1024 of 64   1804 / 2563 / 2974 against 1938 / 2689 / 3033
//   F 1408 of 64; D 4096, F 4096 of 16, F 14336 of 8      3424; 5368, 17088 against 3057; 4896, 15710
//   3000 tokens, the same six                             895 / 1302 / 1356, 1670, 2445, 7089 against
//                                                         991 / 1303 / 1365, 1614, 2340, 6489
//   75 rows an expert, F 14336; 37, F 2048 and 4096       2147; 261, 994 against 2080; 265, 1009
// and by a popularity law of exponent 1.2 (the largest has a fifth of the rows):
//   512 rows an expert on average, F 512 / 768 of 128     2005 / 2850 against 1995 / 2744
//   1024, D 2048, F 1024 of 64; D 1024, F 1024 of 32;     3335; 1013;
//   D 4096, F 1024 of 16                                  1729 against 3020; 921; 1597
constexpr int kMappedGradientMaxF = 1024, kMappedGradientRows = 64, kMappedGradientMaxRows = 768;
bool gradients_in_place(const Args& a) {
  const int64_t pairs = (int64_t)a.T * a.K;
  return in_token_order(a) && ((a.F <= kMappedGradientMaxF && pairs <= (int64_t)kMappedGradientMaxRows * a.E) ||
                               pairs < (int64_t)kMappedGradientRows * a.E);
}

struct Saved {
  int32_t *idx, *counts, *offsets, *perm, *inv_perm;
  float *w, *logits;
  void *xn, *xe, *ye, *g, *u, *h, *gs, *us;
  int64_t total;
};
Saved carve_saved(const Args& a, void* base) {
  Carver c{static_cast<uint8_t*>(base)};
  const int64_t R = rows_of(a), sz = elem_size(a.act_dtype);
  const bool mapped = in_token_order(a);
  Saved s;
  s.idx = static_cast<int32_t*>(c.take((int64_t)a.T * a.K * 4));
  s.w = static_cast<float*>(c.take((int64_t)a.T * a.K * 4));
  s.logits = static_cast<float*>(c.take((int64_t)a.T * a.E * 4));
  s.counts = static_cast<int32_t*>(c.take((int64_t)a.E * 4));
  s.offsets = static_cast<int32_t*>(c.take((int64_t)(a.E + 1) * 4));
  s.perm = static_cast<int32_t*>(c.take(R * 4));
  s.inv_perm = static_cast<int32_t*>(c.take((int64_t)a.T * a.K * 4));
  s.xn = a.normed ? c.take((int64_t)a.T * a.D * sz) : nullptr;
  s.xe = mapped ? nullptr : c.take(R * a.D * sz);
  // (the backward pass reads them for the gradients of weights on the output, in token order not even for those)
  s.ye = mapped || a.scale_input ? nullptr : c.take(R * a.D * sz);
  const bool keep = !streams(a);
  s.g = keep ? c.take(R * a.F * sz) : nullptr;
  s.u = keep ? c.take(R * a.F * sz) : nullptr;
  s.h = mapped ? c.take(R * a.F * sz) : nullptr;
  s.gs = a.F_shared > 0 ? c.take((int64_t)a.T * a.F_shared * sz) : nullptr;
  s.us = a.F_shared > 0 ? c.take((int64_t)a.T * a.F_shared * sz) : nullptr;
  s.total = c.used;
  return s;
}

struct ForwardScratch {
  void *disp, *router, *h, *hs, *ye;
  int64_t disp_bytes, router_bytes, total;
};
ForwardScratch carve_forward(const Args& a, void* base) {
  Carver c{static_cast<uint8_t*>(base)};
  const int64_t sz = elem_size(a.act_dtype);
  ForwardScratch f;
  f.disp_bytes = fs2moe_dispatch_workspace_bytes(a.T, a.K, a.E);
  f.disp = c.take(f.disp_bytes);
  f.router_bytes = fs2moe_router_workspace_bytes(a.T, a.D, a.E, a.act_dtype);
  f.router = f.router_bytes > 0 ? c.take(f.router_bytes) : nullptr;
  f.h = in_token_order(a) ? nullptr : c.take(rows_of(a) * a.F * sz);
  f.hs = a.F_shared > 0 ? c.take((int64_t)a.T * a.F_shared * sz) : nullptr;
  f.ye = in_token_order(a) || a.scale_input ? c.take(rows_of(a) * a.D * sz) : nullptr;
  f.total = c.used;
  return f;
}

struct BackwardScratch {
  void *xe, *dye, *dh, *dg, *du, *dxe, *dl, *router, *d_router, *dx_router, *dhs, *dgs, *dus, *dx_shared, *dxn,
      *norm, *part, *part_shared;
  float* d_w;
  int64_t norm_bytes, total;
};
// the weight gradients of a step, with the buffers they are computed from
int requests(const Args& a, const Saved& s, const BackwardScratch& b, WgradRequest* r) {
  const int Ep = padded_experts(a);
  const void* x = a.normed ? s.xn : a.x;
  int n = 0;
  // (wanted or not goes by the caller's pointer: the buffers' are null while the sizes are taken)
  auto add = [&](void* dw, const void* left, const void* right, int M, int N, bool grouped, bool map_a = false,
                 bool map_b = false) {
    if (dw != nullptr) r[n++] = WgradRequest{left, right, dw, M, N, grouped, 1, map_a, map_b};
  };
  const bool mapped = gradients_in_place(a);
  const void* xe = mapped ? x : in_token_order(a) ? b.xe : s.xe;
  add(a.d_gate, xe, b.dg, a.D, a.F, true, mapped);
  add(a.d_up, xe, b.du, a.D, a.F, true, mapped);
  add(a.d_down, b.dh, mapped ? a.dout : b.dye, a.F, a.D, true, false, mapped);  // (dh holds h by then)
  if (a.F_shared > 0) {
    add(a.d_shared_gate, b.dgs, x, a.F_shared, a.D, false);
    add(a.d_shared_up, b.dus, x, a.F_shared, a.D, false);
    add(a.d_shared_down, a.dout, b.dhs, a.D, a.F_shared, false);
  }
  add(a.d_router, x, b.dl, a.D, Ep, false);
  if (a.d_router != nullptr && Ep != a.E) r[n - 1].dw = b.d_router;
  return n;
}
bool beside(const Args& a, bool backward) {
  return a.F_shared > 0 && a.T > 16 &&
         branch_pays(a.T, a.K, a.E, a.D, a.F, a.F_shared, a.act_dtype, a.act_dtype, true, backward);
}

BackwardScratch carve_backward(const Args& a, void* base) {
  Carver c{static_cast<uint8_t*>(base)};
  const int64_t R = rows_of(a), sz = elem_size(a.act_dtype), T = a.T;
  const int Ep = padded_experts(a);
  BackwardScratch b;
  // (in token order for the weight gradients alone, and only for those that are asked for)
  const bool copies = !gradients_in_place(a), mapped = in_token_order(a);
  b.xe = copies && mapped && (a.d_gate != nullptr || a.d_up != nullptr) ? c.take(R * a.D * sz) : nullptr;
  b.dye = copies && (!mapped || a.d_down != nullptr) ? c.take(R * a.D * sz) : nullptr;
  b.dh = c.take(R * a.F * sz);
  b.dg = c.take(R * a.F * sz);
  b.du = c.take(R * a.F * sz);
  b.dxe = c.take(R * a.D * sz);
  b.d_w = static_cast<float*>(c.take(T * a.K * 4));
  b.dl = c.take(T * Ep * sz);
  b.router = Ep != a.E ? c.take((int64_t)a.D * Ep * sz) : nullptr;
  b.d_router = Ep != a.E ? c.take((int64_t)a.D * Ep * sz) : nullptr;
  b.dx_router = c.take(T * a.D * sz);
  const int64_t sh = T * a.F_shared * sz;
  b.dhs = a.F_shared > 0 ? c.take(sh) : nullptr;
  b.dgs = a.F_shared > 0 ? c.take(sh) : nullptr;
  b.dus = a.F_shared > 0 ? c.take(sh) : nullptr;
  b.dx_shared = a.F_shared > 0 ? c.take(T * a.D * sz) : nullptr;
  b.dxn = a.normed ? c.take(T * a.D * sz) : nullptr;
  b.norm_bytes = a.normed ? fs2moe_rms_norm_backward_workspace_bytes(a.T, a.D) : 0;
  b.norm = a.normed ? c.take(b.norm_bytes) : nullptr;
  WgradRequest r[8];
  const int n = requests(a, Saved{}, b, r);
  // (the weight gradients' partial sums, after those of the rows' gradients)
  int64_t part = wgrad_plan(r, n, a.E, planned_rows(a), T, a.act_dtype);
  auto parts = [&](int64_t rows, int64_t planned, int E, int F) {
    const int n = split_parts(2, planned, E, F, a.D, a.act_dtype);
    return n > 1 ? (int64_t)n * rows * a.D * 4 : 0;
  };
  const bool want_x = a.dx != nullptr || a.d_norm_weight != nullptr;
  if (want_x || (a.scale_input && a.d_router != nullptr)) part = std::max(part, parts(R, planned_rows(a), a.E, a.F));
  // (the shared expert's have a place of their own where they may be at work beside the others)
  const int64_t part_shared = want_x && a.F_shared > 0 ? parts(T, T, 0, a.F_shared) : 0;
  const bool apart = beside(a, true);
  b.part = c.take(apart ? part : std::max(part, part_shared));
  b.part_shared = apart ? c.take(part_shared) : b.part;
  b.total = c.used;
  return b;
}

bool sizes_ok(const Args& a) {
  return a.T >= 0 && a.D >= 8 && a.F >= 8 && a.E >= 1 && a.E <= FS2MOE_MAX_EXPERTS && a.K >= 1 && a.K <= a.E &&
         a.K <= FS2MOE_MAX_TOP_K && a.F_shared >= 0 && a.tile_m >= 1 && a.D % 8 == 0 && a.F % 8 == 0 &&
         a.F_shared % 8 == 0 && (a.act_dtype == FS2MOE_F32 || a.act_dtype == FS2MOE_BF16) &&
         rows_of(a) < (1ll << 31) && swiglu_train_applies(a.act_dtype, a.D, a.F, rows_of(a)) &&
         (a.F_shared == 0 || swiglu_train_applies(a.act_dtype, a.D, a.F_shared, a.T)) &&
         swiglu_train_applies(a.act_dtype, a.D, padded_experts(a), a.T);
}
// What the stage calls ask of their operands, before anything is launched: the kernels behind the pieces
// that are called directly (swiglu_train, gemm_sum, wgrad_all) move 16 bytes at a time.
int check(const Args* a, int64_t saved, int64_t scratch) {
  FS2_REQUIRE(a->x && a->router && a->w_gate && a->w_up && a->w_down && a->saved && a->workspace,
              "train: null pointer");
  FS2_REQUIRE((a->F_shared > 0) == (a->shared_gate && a->shared_up && a->shared_down),
              "train: the shared expert needs its three matrices and F_shared > 0");
  FS2_REQUIRE(a->saved_bytes >= saved && a->workspace_bytes >= scratch,
              "train: buffers of %lld and %lld bytes are smaller than the %lld and %lld needed",
              (long long)a->saved_bytes, (long long)a->workspace_bytes, (long long)saved, (long long)scratch);
  FS2_REQUIRE(((reinterpret_cast<uintptr_t>(a->saved) | reinterpret_cast<uintptr_t>(a->workspace)) & 255u) == 0,
              "train: buffers must be 256-byte aligned");
  FS2_REQUIRE(aligned16(a->w_gate) && aligned16(a->w_up) && aligned16(a->w_down) && aligned16(a->shared_gate) &&
                  aligned16(a->shared_up) && aligned16(a->shared_down),
              "train: weights must be 16-byte aligned");
  // (rows that are normalised are read by the router alone, which looks at their address itself)
  FS2_REQUIRE(a->normed || aligned16(a->x), "train: x must be 16-byte aligned");
  return FS2MOE_OK;
}
}  // namespace
}  // namespace fs2moe

using namespace fs2moe;

extern "C" int64_t fs2moe_train_saved_bytes(const fs2moe_train_args* a) {
  return a != nullptr && sizes_ok(*a) ? carve_saved(*a, nullptr).total : -1;
}

extern "C" int64_t fs2moe_train_workspace_bytes(const fs2moe_train_args* a, int32_t backward) {
  if (a == nullptr || !sizes_ok(*a)) return -1;
  return backward ? carve_backward(*a, nullptr).total : carve_forward(*a, nullptr).total;
}

extern "C" int fs2moe_train_forward(const fs2moe_train_args* a, void* stream) {
  FS2_REQUIRE(a != nullptr && sizes_ok(*a), "train_forward: sizes this call does not take");
  if (a->T == 0) return FS2MOE_OK;
  const Saved s = carve_saved(*a, a->saved);
  const ForwardScratch f = carve_forward(*a, a->workspace);
  if (int rc = check(a, s.total, f.total)) return rc;
  FS2_REQUIRE(a->out && a->router_read, "train_forward: null pointer");
  FS2_REQUIRE(aligned16(a->out) && aligned16(a->residual), "train_forward: out and residual must be 16-byte aligned");
  const int64_t R = rows_of(*a);
  const void* x = a->normed ? s.xn : a->x;
  Branch branch(beside(*a, false), stream);
  auto shared = [&]() -> int {
    if (int rc = branch.fork()) return rc;
    return swiglu_train(x, nullptr, nullptr, nullptr, 0, a->shared_gate, a->shared_up, a->shared_down, a->D,
                        a->F_shared, a->T, a->T, a->act_dtype, s.gs, s.us, f.hs, a->out, branch.stream());
  };
  int rc;
  if (branch.beside() && !a->normed && (rc = shared())) return rc;
  // (rows that stay in token order need no copy: the router's last kernel counts for the dispatch, a launch fewer; 4096
  // tokens, top-8 of 128, D 2048, F 768 1580 -> 1573 us, 4444, D 1280, F 704 1094 -> 1087)
  DispatchAfterRouter disp{a->tile_m, R, s.counts, s.offsets, s.perm, s.inv_perm, f.disp, f.disp_bytes, nullptr, nullptr, false};
  rc = router_then_dispatch(a->x, a->normed ? a->norm_weight : nullptr, a->normed ? a->norm_eps : 0.f,
                                a->normed ? s.xn : nullptr, a->router_read, a->router_bias, a->T, a->D, a->E, a->K,
                                a->act_dtype, a->score_fn, a->renormalize, s.idx, s.w, s.logits, f.router,
                                f.router_bytes, s.xe == nullptr ? &disp : nullptr, stream);
  if (rc) return rc;
  if (branch.beside() && a->normed && (rc = shared())) return rc;
  if (!disp.done &&
      (rc = fs2moe_dispatch(s.idx, s.w, x, a->T, a->K, a->E, a->D, a->tile_m, a->act_dtype, a->scale_input, R,
                            s.counts, s.offsets, s.perm, s.inv_perm, s.xe, f.disp, f.disp_bytes, stream)))
    return rc;
  const bool mapped = in_token_order(*a);
  void* ye = s.ye != nullptr ? s.ye : f.ye;
  if (s.g == nullptr)
    rc = grouped_swiglu_planned(s.xe, nullptr, s.counts, s.offsets, a->w_gate, a->w_up, a->w_down, nullptr, nullptr,
                                nullptr, a->E, a->D, a->F, R, planned_rows(*a), a->act_dtype, a->act_dtype, f.h, ye,
                                a->T, stream);
  else
    rc = swiglu_train(mapped ? x : s.xe, mapped ? s.perm : nullptr, s.counts, s.offsets, a->E, a->w_gate, a->w_up,
                      a->w_down, a->D, a->F, R, planned_rows(*a), a->act_dtype, s.g, s.u, mapped ? s.h : f.h, ye,
                      stream);
  if (rc) return rc;
  if ((rc = branch.join())) return rc;
  if (a->F_shared > 0 && !branch.beside() && (rc = shared())) return rc;
  const void* base = a->F_shared > 0 ? a->out : nullptr;
  if (a->residual != nullptr)
    return fs2moe_combine_residual(ye, s.inv_perm, s.idx, s.w, base, a->residual, a->T, a->K, a->D,
                                   a->act_dtype, a->scale_input ? 0 : 1, a->out, stream);
  return fs2moe_combine(ye, s.inv_perm, s.idx, s.w, base, a->T, a->K, a->D, a->act_dtype,
                        a->scale_input ? 0 : 1, a->out, stream);
}

extern "C" int fs2moe_train_backward(const fs2moe_train_args* a, void* stream) {
  FS2_REQUIRE(a != nullptr && sizes_ok(*a), "train_backward: sizes this call does not take");
  if (a->T == 0) return FS2MOE_OK;
  const Saved s = carve_saved(*a, a->saved);
  const BackwardScratch b = carve_backward(*a, a->workspace);
  if (int rc = check(a, s.total, b.total)) return rc;
  const bool want_x = a->dx != nullptr || a->d_norm_weight != nullptr;
  FS2_REQUIRE(a->dout && aligned16(a->dout), "train_backward: dout must be 16-byte aligned");
  FS2_REQUIRE(!(a->normed && want_x) || (aligned16(a->x) && aligned16(a->norm_weight)),
              "train_backward: x and the norm's weight must be 16-byte aligned");
  FS2_REQUIRE(!want_x || padded_experts(*a) != a->E || aligned16(a->router),
              "train_backward: router must be 16-byte aligned");
  // (a padded router gradient is copied out element by element)
  for (const void* p : {a->dx, padded_experts(*a) == a->E ? a->d_router : nullptr, a->d_gate, a->d_up, a->d_down,
                        a->d_shared_gate, a->d_shared_up, a->d_shared_down, a->d_norm_weight})
    FS2_REQUIRE(aligned16(p), "train_backward: gradients must be 16-byte aligned");
  FS2_REQUIRE(a->d_norm_weight == nullptr || (a->normed && a->norm_weight != nullptr),
              "train_backward: a gradient of a norm weight that is not there");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int T = a->T, D = a->D, E = a->E, K = a->K, F = a->F, Fs = a->F_shared, dt = a->act_dtype;
  const int Ep = padded_experts(*a), score_fn = a->score_fn & ~FS2MOE_ROUTER_OUT_IN;
  const int64_t R = rows_of(*a);
  const void* x = a->normed ? s.xn : a->x;
  int rc;
  // the shared expert, which depends on what the forward pass kept and on dout only
  Branch branch(beside(*a, true), stream);
  auto shared = [&]() -> int {
    if (int rc = branch.fork()) return rc;
    void* on = branch.stream();
    if (int rc = fs2moe_grouped_gemm(a->dout, nullptr, nullptr, nullptr, a->shared_down, FS2MOE_W_IN_OUT, 1, D, Fs, T, dt,
                                     b.dhs, on))
      return rc;
    if (int rc = fs2moe_swiglu_backward(s.gs, s.us, b.dhs, T, Fs, dt, b.dhs, b.dgs, b.dus, on)) return rc;
    if (!want_x) return FS2MOE_OK;
    return gemm_sum(b.dgs, a->shared_gate, b.dus, a->shared_up, FS2MOE_W_IN_OUT, nullptr, nullptr, 0, Fs, D, T, T, dt,
                    b.dx_shared, b.part_shared, on);
  };
  if (branch.beside() && (rc = shared())) return rc;
  // rows in expert order: the output gradients, with those of output-side weights that are applied to them, and in
  // token order the copies for the weight gradients
  const bool mapped = in_token_order(*a);
  auto gather = [&](const void* rows, void* to, bool weighted) -> int {
    const dim3 grid((unsigned)(((int64_t)T * K + 3) / 4)), block(256);
    if (dt == FS2MOE_BF16)
      hipLaunchKernelGGL(gather_backward_kernel<uint16_t>, grid, block, 0, st, static_cast<const uint16_t*>(rows),
                         static_cast<const uint16_t*>(s.ye), s.inv_perm, s.w, T * K, K, D, weighted,
                         static_cast<uint16_t*>(to), b.d_w);
    else
      hipLaunchKernelGGL(gather_backward_kernel<float>, grid, block, 0, st, static_cast<const float*>(rows),
                         static_cast<const float*>(s.ye), s.inv_perm, s.w, T * K, K, D, weighted,
                         static_cast<float*>(to), b.d_w);
    return check_launch("gather_backward");
  };
  if (b.dye != nullptr && (rc = gather(a->dout, b.dye, !a->scale_input && !mapped))) return rc;
  if (b.xe != nullptr && (rc = gather(x, b.xe, false))) return rc;
  // the experts: dh, then h, dg and du, then the rows' gradient
  const int64_t planned = planned_rows(*a);
  if ((rc = grouped_gemm_planned(b.dye != nullptr ? b.dye : a->dout, b.dye != nullptr ? nullptr : s.perm, s.counts,
                                 s.offsets, a->w_down, FS2MOE_W_OUT_IN, E, D, F, R, planned, dt, b.dh, stream)))
    return rc;
  const void *g = s.g, *u = s.u;
  if (g == nullptr) {
    if ((rc = grouped_gemm_planned(s.xe, nullptr, s.counts, s.offsets, a->w_gate, FS2MOE_W_IN_OUT, E, D, F, R, planned,
                                   dt, b.dg, stream)) ||
        (rc = grouped_gemm_planned(s.xe, nullptr, s.counts, s.offsets, a->w_up, FS2MOE_W_IN_OUT, E, D, F, R, planned,
                                   dt, b.du, stream)))
      return rc;
    g = b.dg;
    u = b.du;
  }
  if (mapped) {
    const uint16_t* dh = static_cast<const uint16_t*>(b.dh);
    hipLaunchKernelGGL(swiglu_backward_pairs_kernel, dim3((unsigned)(((int64_t)T * K + 3) / 4)), dim3(256), 0, st,
                       static_cast<const uint16_t*>(g), static_cast<const uint16_t*>(u),
                       static_cast<const uint16_t*>(s.h), dh, s.inv_perm, s.w, T * K, F,
                       static_cast<uint16_t*>(b.dh), static_cast<uint16_t*>(b.dg), static_cast<uint16_t*>(b.du),
                       b.d_w);
    rc = check_launch("swiglu_backward_pairs");
  } else {
    rc = fs2moe_swiglu_backward(g, u, b.dh, R, F, dt, b.dh, b.dg, b.du, stream);
  }
  if (rc) return rc;
  if (want_x || (a->scale_input && a->d_router != nullptr))
    if ((rc = gemm_sum(b.dg, a->w_gate, b.du, a->w_up, FS2MOE_W_OUT_IN, s.counts, s.offsets, E, F, D, R, planned,
                       dt, b.dxe, b.part, stream)))
      return rc;
  // combine weights -> logits
  if (want_x || a->d_router != nullptr) {
    if (a->scale_input && (rc = fs2moe_pair_dot(b.dxe, nullptr, s.inv_perm, x, T, K, D, dt, b.d_w, stream))) return rc;
    if ((rc = router_backward_ld(s.logits, s.idx, s.w, b.d_w, T, E, K, score_fn, a->renormalize, dt, b.dl, Ep, stream)))
      return rc;
  }
  if ((rc = branch.join())) return rc;
  if (Fs > 0 && !branch.beside() && (rc = shared())) return rc;
  // all weight gradients
  WgradRequest r[8];
  const int n = requests(*a, s, b, r);
  if (n > 0) {
    (void)wgrad_plan(r, n, E, planned, T, dt);
    if ((rc = wgrad_all(r, n, gradients_in_place(*a) ? s.perm : nullptr, s.counts, s.offsets, E, R, T, dt, b.part,
                        stream)))
      return rc;
    if (a->d_router != nullptr && Ep != E && (rc = copy_columns(b.d_router, Ep, a->d_router, E, D, dt, st))) return rc;
  }
  if (!want_x) return FS2MOE_OK;
  // the rows: through the router, the shared expert and (scattered back) the experts
  const void* router = a->router;
  if (Ep != E) {
    if ((rc = copy_columns(a->router, E, b.router, Ep, D, dt, st))) return rc;
    router = b.router;
  }
  if ((rc = fs2moe_grouped_gemm(b.dl, nullptr, nullptr, nullptr, router, FS2MOE_W_OUT_IN, 1, Ep, D, T, dt,
                                b.dx_router, stream)))
    return rc;
  void* dx = a->normed ? b.dxn : a->dx;
  rc = Fs > 0 ? fs2moe_combine_residual(b.dxe, s.inv_perm, s.idx, s.w, b.dx_router, b.dx_shared, T, K, D, dt,
                                        a->scale_input ? 1 : 0, dx, stream)
              : fs2moe_combine(b.dxe, s.inv_perm, s.idx, s.w, b.dx_router, T, K, D, dt, a->scale_input ? 1 : 0, dx,
                               stream);
  if (rc || !a->normed) return rc;
  // (dxe's buffer is free by now: where only the norm weight's gradient is wanted, the rows' goes there)
  return fs2moe_rms_norm_backward(a->x, a->norm_weight, a->norm_eps, b.dxn, T, D, dt,
                                  a->dx != nullptr ? a->dx : b.dxe, a->d_norm_weight, b.norm, b.norm_bytes, stream);
}
