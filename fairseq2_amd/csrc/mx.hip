// W8A8 expert path: block-scaled e4m3 activations against e4m3 weights on the fp8 matrix pipe.
// Host side of experts_mx.h.  No counterpart in the reference (its experts run in the parameters'
// dtype, experts.py:102-112); an opt-in of this library.
#include "experts_half.h"
#include "experts_mx.h"

namespace fs2moe {
// x [T, D] bf16 -> e4m3 codes [T, D] and one scale byte per row and 32 features, k-group major:
// [D / 128][T][4].  A lane owns a block of 32 features (64 bytes in, 32 bytes out); consecutive
// lanes take consecutive blocks of a row, so four lanes fill a scale dword.
__global__ __launch_bounds__(256) void mx_quantize_kernel(const uint16_t* __restrict__ x, int64_t T,
                                                          int D, uint8_t* __restrict__ xq,
                                                          uint8_t* __restrict__ xs) {
  const int lane = threadIdx.x & 63;
  const int64_t wave = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int nb = D / 32;
  const int64_t blocks = T * nb;
  for (int64_t b = wave * 64 + lane; b < blocks; b += (int64_t)gridDim.x * 256) {
    const uint16_t* src = x + b * 32;
    u32x4 in[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) in[j] = *reinterpret_cast<const u32x4*>(src + 8 * j);
    float v[32];
    float amax = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[8 * j + 2 * i] = __uint_as_float(in[j][i] << 16);
        v[8 * j + 2 * i + 1] = __uint_as_float(in[j][i] & 0xffff0000u);
        amax = fmaxf(amax, fmaxf(fabsf(v[8 * j + 2 * i]), fabsf(v[8 * j + 2 * i + 1])));
      }
    const int X = mx::block_exponent(amax);
    const float inv = __builtin_ldexpf(1.0f, -X);
    u32x4 out[2];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      out[j >> 2][j & 3] = mx::to_e4m3x4(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3], inv);
    *reinterpret_cast<u32x4*>(xq + b * 32) = out[0];
    *reinterpret_cast<u32x4*>(xq + b * 32 + 16) = out[1];
    const int64_t row = b / nb;
    const int kb = (int)(b - row * nb);
    xs[((int64_t)(kb >> 2) * T + row) * 4 + (kb & 3)] = (uint8_t)(X + 127);
  }
}
}  // namespace fs2moe

using namespace fs2moe;

static int mx_cu_count() {
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

extern "C" int fs2moe_mx_quantize(const void* x, int64_t rows, int32_t D, void* codes, void* scales,
                                  void* stream) {
  FS2_REQUIRE(x && codes && scales, "mx_quantize: null pointer");
  FS2_REQUIRE(rows >= 0 && D > 0 && D % 128 == 0, "mx_quantize: rows=%lld, D=%d (a multiple of 128)",
              (long long)rows, D);
  FS2_REQUIRE(aligned16(x) && aligned16(codes), "mx_quantize: buffers must be 16-byte aligned");
  if (rows == 0) return FS2MOE_OK;
  const int64_t blocks32 = rows * (D / 32);
  int64_t grid = (blocks32 + 255) / 256;
  if (grid > 8192) grid = 8192;
  hipLaunchKernelGGL(mx_quantize_kernel, dim3((unsigned)grid), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(x), rows, D,
                     static_cast<uint8_t*>(codes), static_cast<uint8_t*>(scales));
  return check_launch("mx_quantize");
}

extern "C" int fs2moe_grouped_swiglu_w8a8_supported(int32_t D, int32_t F, int64_t max_rows) {
  const int64_t wide = D > F ? D : F;
  return (D > 0 && F > 0 && D % mx::UK == 0 && F % mx::UK == 0 && max_rows >= 0 &&
          max_rows * wide <= 0xffffffffll && (int64_t)D * F <= 0xffffffffll)
             ? 1
             : 0;
}

int fs2moe::grouped_swiglu_w8a8_planned(const void* xq, const void* xs, const int32_t* row_map, const int32_t* counts,
                                        const int32_t* offsets, const void* w_gate, const void* w_up,
                                        const void* w_down, const float* s_gate, const float* s_up,
                                        const float* s_down, int32_t E, int32_t D, int32_t F, int64_t x_rows,
                                        int64_t max_rows, int64_t planned, void* hq, void* hs, void* ye,
                                        void* stream) {
  using namespace mx;
  FS2_REQUIRE(xq && xs && counts && offsets && w_gate && w_up && w_down && s_gate && s_up && s_down &&
                  hq && hs && ye,
              "grouped_swiglu_w8a8: null pointer");
  FS2_REQUIRE(E >= 1 && E <= FS2MOE_MAX_EXPERTS, "grouped_swiglu_w8a8: E=%d outside [1, %d]", E,
              FS2MOE_MAX_EXPERTS);
  FS2_REQUIRE(max_rows >= 0 && max_rows < (1ll << 31), "grouped_swiglu_w8a8: max_rows=%lld",
              (long long)max_rows);
  // x_rows: the rows of xq / xs (their number places a k-group's scales): the token count with a
  // row map, else max_rows
  FS2_REQUIRE(x_rows >= 1 && x_rows < (1ll << 31) && (row_map != nullptr || x_rows == max_rows),
              "grouped_swiglu_w8a8: x_rows=%lld", (long long)x_rows);
  FS2_REQUIRE(fs2moe_grouped_swiglu_w8a8_supported(D, F, max_rows),
              "grouped_swiglu_w8a8: D=%d and F=%d must be multiples of %d, and the operands "
              "addressable with 32-bit byte offsets",
              D, F, UK);
  FS2_REQUIRE(aligned16(xq) && aligned16(w_gate) && aligned16(w_up) && aligned16(w_down) &&
                  aligned16(hq) && aligned16(ye) && aligned16(s_gate) && aligned16(s_up) &&
                  aligned16(s_down) && (reinterpret_cast<uintptr_t>(xs) & 3u) == 0 &&
                  (reinterpret_cast<uintptr_t>(hs) & 3u) == 0,
              "grouped_swiglu_w8a8: buffers must be 16-byte aligned (scale bytes: 4)");
  if (max_rows == 0) return FS2MOE_OK;
  FS2_REQUIRE(x_rows * (int64_t)D <= 0xffffffffll, "grouped_swiglu_w8a8: xq is addressed with 32-bit byte offsets");
  hipStream_t st = static_cast<hipStream_t>(stream);
  Groups g{counts, offsets, E, 0, (int)planned};
  g.once_past_cache = weights_past_cache(E, pairs_of(g, max_rows), D, F, 1);
  // (us without and with, loaded evenly and by a popularity law: 1100 tokens, top-8 of 128, D 2048, F 768 181, 172 and 170,
  // 166; 2000 202, 193 and 215, 214; 1100, top-2 of 16, D 4096, F 4096 219, 208 and 278, 275)
  const bool once = g.once_past_cache && pairs_of(g, max_rows) <= kOnceRows * E;
  auto k1 = once ? glu_gemm_mx_kernel<true, true> : glu_gemm_mx_kernel<true>;
  auto k2 = once ? glu_gemm_mx_kernel<false, true> : glu_gemm_mx_kernel<false>;
  static bool attr_set = false;  // benign race: setting the attribute is idempotent
  if (!attr_set) {
    for (const void* k : {reinterpret_cast<const void*>(glu_gemm_mx_kernel<true>),
                          reinterpret_cast<const void*>(glu_gemm_mx_kernel<false>),
                          reinterpret_cast<const void*>(glu_gemm_mx_kernel<true, true>),
                          reinterpret_cast<const void*>(glu_gemm_mx_kernel<false, true>)}) {
      hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM_BYTES);
      if (e != hipSuccess) {
        set_error("grouped_swiglu_w8a8: cannot reserve %d bytes of LDS: %s", SMEM_BYTES,
                  hipGetErrorString(e));
        return FS2MOE_ERR_LAUNCH;
      }
    }
    attr_set = true;
  }
  const int num_blocks = mx_cu_count();
  if (num_blocks == 0) {
    set_error("grouped_swiglu_w8a8: cannot query the compute-unit count");
    return FS2MOE_ERR_LAUNCH;
  }
  const int nt1 = (F + 127) / 128, nt2 = (D + 255) / 256;
  {
    const int64_t m_tiles = max_rows / BM + E + 1;
    if (m_tiles * nt1 > 0x7fffffffll || m_tiles * nt2 > 0x7fffffffll) {
      set_error("grouped_swiglu_w8a8: too many tiles");
      return FS2MOE_ERR_UNSUPPORTED;
    }
  }
  // Few tiles: the smaller tiles of experts_half.h (the same bits).
  auto half = [&](auto bm_c, auto dual_c, const void* a, const void* as, const int32_t* map, int K, const void* b0,
                  const void* b1, const float* s0, const float* s1, void* c, void* cs, int N, int64_t a_rows,
                  int64_t c_rows, const char* what) -> int {
    constexpr int HBM = decltype(bm_c)::value, HBN = 128;
    constexpr bool DUAL = decltype(dual_c)::value;
    constexpr int bytes = half_tiles::smem_bytes(HBM, HBN, half_tiles::W_MX), bn = DUAL ? HBN / 2 : HBN;
    auto shared = glu_gemm_half_kernel<HBM, HBN, DUAL, half_tiles::W_MX>;
    auto past = glu_gemm_half_kernel<HBM, HBN, DUAL, half_tiles::W_MX, false, false, true>;
    static bool half_attr_set = false;  // benign race: setting the attribute is idempotent
    if (!half_attr_set) {
      for (const void* k : {reinterpret_cast<const void*>(shared), reinterpret_cast<const void*>(past)}) {
        hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        if (e != hipSuccess) {
          set_error("%s: cannot reserve %d bytes of LDS: %s", what, bytes, hipGetErrorString(e));
          return FS2MOE_ERR_LAUNCH;
        }
      }
      half_attr_set = true;
    }
    auto k = g.once_past_cache && pairs_of(g, max_rows) / E <= half_tiles::once_rows(HBM) ? past : shared;
    hipLaunchKernelGGL(k, dim3((unsigned)num_blocks), dim3(half_tiles::THREADS), bytes, st,
                       static_cast<const uint8_t*>(a), map, K, static_cast<const uint8_t*>(b0),
                       static_cast<const uint8_t*>(b1), s0, s1, static_cast<uint8_t*>(c), N, K, N, g,
                       (N + bn - 1) / bn,
                       HalfMx{static_cast<const uint8_t*>(as), static_cast<uint8_t*>(cs), (int)a_rows, (int)c_rows});
    return check_launch(what);
  };
  using I64 = std::integral_constant<int, 64>;
  using I128 = std::integral_constant<int, 128>;
  const bool counted = (max_rows / 64 + E + 1) * (((D > F ? D : F) + 63) / 64) <= 0x7fffffffll;
  auto pick = [&](bool dual, int K, int N) {
    return counted ? half_tiles::pick(dual, false, g.rows_to_plan(max_rows), E, K / 2, N, num_blocks) : 0;
  };
  const char* what = "glu_gemm_mx<gate,up>";
  int rc;
  switch (pick(true, D, F)) {
    case 2:
      rc = half(I64{}, std::true_type{}, xq, xs, row_map, D, w_gate, w_up, s_gate, s_up, hq, hs, F, x_rows, max_rows, what);
      break;
    case 3:
      rc = half(I128{}, std::true_type{}, xq, xs, row_map, D, w_gate, w_up, s_gate, s_up, hq, hs, F, x_rows, max_rows, what);
      break;
    default:
      hipLaunchKernelGGL(k1, dim3((unsigned)num_blocks), dim3(NWAVES * 64), SMEM_BYTES, st,
                         static_cast<const uint8_t*>(xq), static_cast<const uint8_t*>(xs), row_map,
                         static_cast<const uint8_t*>(w_gate), static_cast<const uint8_t*>(w_up), s_gate, s_up, hq,
                         static_cast<uint8_t*>(hs), F, D, F, g, nt1, (int)x_rows, (int)max_rows);
      rc = check_launch(what);
  }
  if (rc) return rc;
  what = "glu_gemm_mx<down>";
  switch (pick(false, F, D)) {
    case 2:
      return half(I64{}, std::false_type{}, hq, hs, nullptr, F, w_down, nullptr, s_down, nullptr, ye, nullptr, D, max_rows, 0, what);
    case 3:
      return half(I128{}, std::false_type{}, hq, hs, nullptr, F, w_down, nullptr, s_down, nullptr, ye, nullptr, D, max_rows, 0, what);
  }
  hipLaunchKernelGGL(k2, dim3((unsigned)num_blocks), dim3(NWAVES * 64), SMEM_BYTES, st,
                     static_cast<const uint8_t*>(hq), static_cast<const uint8_t*>(hs),
                     static_cast<const int32_t*>(nullptr), static_cast<const uint8_t*>(w_down),
                     static_cast<const uint8_t*>(nullptr), s_down, static_cast<const float*>(nullptr),
                     ye, static_cast<uint8_t*>(nullptr), D, F, D, g, nt2, (int)max_rows, 0);
  return check_launch(what);
}

extern "C" int fs2moe_grouped_swiglu_w8a8(const void* xq, const void* xs, const int32_t* row_map,
                                          const int32_t* counts, const int32_t* offsets,
                                          const void* w_gate, const void* w_up, const void* w_down,
                                          const float* s_gate, const float* s_up,
                                          const float* s_down, int32_t E, int32_t D, int32_t F,
                                          int64_t x_rows, int64_t max_rows, void* hq, void* hs,
                                          void* ye, void* stream) {
  return grouped_swiglu_w8a8_planned(xq, xs, row_map, counts, offsets, w_gate, w_up, w_down, s_gate, s_up, s_down, E, D,
                                     F, x_rows, max_rows, 0, hq, hs, ye, stream);
}
