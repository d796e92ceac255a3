// Library-wide pieces of the C ABI: version, thread-local error text, launch checking.
#include <cstdarg>
#include <cstdio>
#include <mutex>

#include "common.h"

namespace fs2moe {

static thread_local char g_error[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s: launch failed: %s", what, hipGetErrorString(e));
    return FS2MOE_ERR_LAUNCH;
  }
  return FS2MOE_OK;
}

}  // namespace fs2moe

extern "C" int fs2moe_abi_version(void) { return FS2MOE_ABI_VERSION; }

extern "C" const char* fs2moe_last_error(void) { return fs2moe::g_error; }

// ---- the whole layer ----------------------------------------------------------------------------
namespace {

// Carves 256-byte aligned pieces out of the caller's workspace (or only adds up their sizes).
struct Carver {
  uint8_t* base;
  int64_t used = 0;
  void* take(int64_t bytes) {
    void* p = base ? base + used : nullptr;
    used += (bytes + 255) / 256 * 256;
    return p;
  }
};

struct ForwardBuffers {
  int32_t *topk_idx, *counts, *offsets, *perm, *inv_perm;
  float* topk_w;
  void *disp_ws, *router_ws, *xn, *xe, *h, *ye, *shared_h;
  // W8A8: the token rows as block-scaled e4m3 (in the place of xe) and the gated product likewise
  // (in the place of h)
  void *xq, *xs, *hq, *hs;
  // a weight per expert row (in the place of xe) where the expert kernels scale the rows themselves
  float* row_w;
  int64_t max_rows, disp_ws_bytes, router_ws_bytes, total;
};

ForwardBuffers carve_forward(void* workspace, int32_t T, int32_t D, int32_t E, int32_t K, int32_t F,
                             int32_t F_shared, int32_t tile_m, int32_t act_dtype, bool need_xe,
                             bool need_xn, bool act_q = false, bool need_row_w = false) {
  const int64_t esz = fs2moe::elem_size(act_dtype);
  ForwardBuffers b;
  b.max_rows = FS2MOE_MAX_ROWS(T, K, E, tile_m);
  b.disp_ws_bytes = fs2moe_dispatch_workspace_bytes(T, K, E);
  Carver c{static_cast<uint8_t*>(workspace)};
  b.topk_idx = static_cast<int32_t*>(c.take((int64_t)T * K * 4));
  b.topk_w = static_cast<float*>(c.take((int64_t)T * K * 4));
  b.counts = static_cast<int32_t*>(c.take((int64_t)E * 4));
  b.offsets = static_cast<int32_t*>(c.take((int64_t)(E + 1) * 4));
  b.perm = static_cast<int32_t*>(c.take(b.max_rows * 4));
  b.inv_perm = static_cast<int32_t*>(c.take((int64_t)T * K * 4));
  b.disp_ws = c.take(b.disp_ws_bytes);
  b.router_ws_bytes = fs2moe_router_workspace_bytes(T, D, E, act_dtype);
  b.router_ws = b.router_ws_bytes > 0 ? c.take(b.router_ws_bytes) : nullptr;
  b.xn = need_xn ? c.take((int64_t)T * D * esz) : nullptr;
  b.xe = need_xe ? c.take(b.max_rows * D * esz) : nullptr;
  // (4 bytes a row where the copy would have taken D elements: the workspace sized with the copy holds it)
  b.row_w = need_row_w ? static_cast<float*>(c.take(b.max_rows * 4)) : nullptr;
  b.xq = b.xs = b.hq = b.hs = nullptr;
  if (act_q) {
    // T rows of D codes and D / 32 scale bytes each: less than the row copy that is not made, so a
    // workspace of fs2moe_forward_workspace_bytes (sized with the copy) holds them
    b.xq = c.take((int64_t)T * D);
    b.xs = c.take((int64_t)T * (D / 32));
  }
  b.h = c.take(b.max_rows * F * esz);
  if (act_q) {
    // max_rows x (F codes + F / 32 scale bytes) inside the bf16 product's place
    b.hq = b.h;
    b.hs = static_cast<uint8_t*>(b.h) + (b.max_rows * F + 255) / 256 * 256;
  }
  b.ye = c.take(b.max_rows * D * esz);
  b.shared_h = F_shared > 0 ? c.take((int64_t)T * F_shared * esz) : nullptr;
  b.total = c.used;
  return b;
}

}  // namespace

extern "C" int64_t fs2moe_forward_workspace_bytes(int32_t T, int32_t D, int32_t E, int32_t K,
                                                  int32_t F, int32_t F_shared, int32_t tile_m,
                                                  int32_t act_dtype) {
  if (T < 0 || D < 1 || E < 1 || K < 1 || F < 1 || F_shared < 0 || tile_m < 1) return -1;
  // sized for the path that copies the rows: which path runs depends on the mode and the types
  return carve_forward(nullptr, T, D, E, K, F, F_shared, tile_m, act_dtype, true, false).total;
}

extern "C" int64_t fs2moe_forward_norm_workspace_bytes(int32_t T, int32_t D, int32_t E, int32_t K,
                                                       int32_t F, int32_t F_shared, int32_t tile_m,
                                                       int32_t act_dtype) {
  if (T < 0 || D < 1 || E < 1 || K < 1 || F < 1 || F_shared < 0 || tile_m < 1) return -1;
  return carve_forward(nullptr, T, D, E, K, F, F_shared, tile_m, act_dtype, true, true).total;
}

namespace fs2moe {

// Streams of the library's own, two per device: one for callers' streams that run their work, one for those that capture
// it, so that a capture never finds another thread's work on the stream.  Default priority, created on the first use of its
// kind on a device and kept (a process with three streams, the caller's among them, runs 5 tokens of D 5120, F 8192, 16
// experts and a shared one in 323.5 us, one with two or four in 320.5: none is there that is not used).
// Callers' streams that are independent stay so: what a side stream waits for, everything behind it on that stream waits
// for too, so a caller's stream gets it only where nothing of another one's is left on it, and a call has it for itself from
// its branch's beginning to its end; another's shared expert then runs on its own stream.  (Handed to whoever came next: of 7
// and 9 pairs of streams that one did not have to wait for the other on, no call on one ended before a call queued on the
// other, which was held up for 40 ms; now on 6 and 6, the side stream being in one queue of the hardware with the others.)
struct SideStream {
  hipStream_t stream = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
  // the caller's stream of the last branch, whose order covers all that is on this one; where its handle is another
  // stream's by now, a branch of that one may wait for what the destroyed one had left to do
  hipStream_t owner = nullptr;
  bool taken = false, tried = false;
};
namespace {
constexpr int kSideDevices = 64;
struct SideStreams {
  SideStream of[2];
};
SideStreams g_side[kSideDevices];
std::mutex g_side_mu;

// The capture that a stream is part of, 0 where it captures nothing.
unsigned long long capture_of(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  if (hipStreamGetCaptureInfo(stream, &status, &id) != hipSuccess) (void)hipGetLastError();
  return status == hipStreamCaptureStatusNone ? 0 : id;
}

// This thread's calls in the relaxed mode of capturing: a capture, its own or another thread's, may forbid them else.
class Relaxed {
 public:
  Relaxed() : set_(hipThreadExchangeStreamCaptureMode(&mode_) == hipSuccess) {
    if (!set_) (void)hipGetLastError();
  }
  Relaxed(const Relaxed&) = delete;
  Relaxed& operator=(const Relaxed&) = delete;
  ~Relaxed() {
    if (set_) (void)hipThreadExchangeStreamCaptureMode(&mode_);
  }

 private:
  hipStreamCaptureMode mode_ = hipStreamCaptureModeRelaxed;
  const bool set_;
};

// Whether all work of a stream is done.
bool idle(hipStream_t stream) {
  const Relaxed relaxed;
  const bool done = hipStreamQuery(stream) == hipSuccess;
  if (!done) (void)hipGetLastError();
  return done;
}

// For a branch of the caller's stream `main`, until given back; null: there is none to have (creation failed once, it would
// order callers' streams, or the caller's stream is one).
SideStream* take_side_stream(hipStream_t main) {
  if (main == hipStreamPerThread) return nullptr;  // (one handle for a stream of each thread)
  int dev = -1, of = -1;
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipGetDevice(&dev) != hipSuccess || hipStreamGetDevice(main, &of) != hipSuccess ||
      hipStreamIsCapturing(main, &status) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  // (the events would be of the current device, which a launch on another one's stream does not need)
  if (dev != of || dev < 0 || dev >= kSideDevices) return nullptr;
  const bool captures = status != hipStreamCaptureStatusNone;
  std::lock_guard<std::mutex> lock(g_side_mu);
  SideStreams& s = g_side[dev];
  SideStream& side = s.of[captures ? 1 : 0];
  if (!side.tried) {
    const Relaxed relaxed;
    side.tried = true;
    if (hipStreamCreateWithFlags(&side.stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&side.fork, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&side.join, hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();  // the failure is handled here: nothing for the next call to find
      side.stream = nullptr;
    }
  }
  if (side.stream == nullptr || side.taken) return nullptr;
  for (const SideStream& one : s.of)  // (one that is not there is no caller's null stream)
    if (one.stream != nullptr && one.stream == main) return nullptr;
  if (captures) {
    // (a stream that a capture has forked to stays part of it until that capture ends, and another stream of the same
    // capture is a chain of nodes of its own)
    const unsigned long long held = capture_of(side.stream);
    if (held != 0 && (side.owner != main || held != capture_of(main))) return nullptr;
  } else if (side.owner != main && !idle(side.stream)) {
    return nullptr;
  }
  side.owner = main;
  side.taken = true;
  return &side;
}
}  // namespace

bool branch_pays(int T, int K, int E, int D, int F, int F_shared, int act_dtype, int w_dtype, bool late, bool backward) {
  const int64_t reached = (int64_t)T * K < E ? (int64_t)T * K : E;
  const double features = 6.0 * D * T * ((double)K * F + F_shared);
  const double weights = 3.0 * D * ((double)reached * F * elem_size(w_dtype) + (double)F_shared * elem_size(act_dtype));
  const double memory_us = weights / 5e6, products_us = 1.6 * features / (act_dtype == FS2MOE_F32 ? 153e6 : 1200e6);
  return backward ? memory_us + 2.0 * products_us >= 200.0 : memory_us + products_us >= (late ? 350.0 : 130.0);
}

Branch::Branch(bool wanted, void* stream) : main_(stream) {
  if (wanted) side_ = take_side_stream(static_cast<hipStream_t>(stream));
}

Branch::~Branch() {
  (void)join();
  if (side_ == nullptr) return;
  std::lock_guard<std::mutex> lock(g_side_mu);
  side_->taken = false;
}

void* Branch::stream() const { return forked_ ? side_->stream : main_; }

int Branch::mark() {
  if (side_ == nullptr) return FS2MOE_OK;
  if (hipEventRecord(side_->fork, static_cast<hipStream_t>(main_)) != hipSuccess) {
    set_error("cannot fork a stream: %s", hipGetErrorString(hipGetLastError()));
    return FS2MOE_ERR_LAUNCH;
  }
  marked_ = true;
  return FS2MOE_OK;
}

int Branch::fork() {
  if (side_ == nullptr) return FS2MOE_OK;
  if (!marked_)
    if (int rc = mark()) return rc;
  if (hipStreamWaitEvent(side_->stream, side_->fork, 0) != hipSuccess) {
    set_error("cannot fork a stream: %s", hipGetErrorString(hipGetLastError()));
    return FS2MOE_ERR_LAUNCH;
  }
  forked_ = true;
  return FS2MOE_OK;
}

int Branch::join() {
  if (!forked_) return FS2MOE_OK;
  forked_ = false;
  if (hipEventRecord(side_->join, side_->stream) != hipSuccess ||
      hipStreamWaitEvent(static_cast<hipStream_t>(main_), side_->join, 0) != hipSuccess) {
    set_error("cannot join a stream: %s", hipGetErrorString(hipGetLastError()));
    return FS2MOE_ERR_LAUNCH;
  }
  return FS2MOE_OK;
}

}  // namespace fs2moe

namespace {

// normed: the rows are RMS-normalised on the way into the router (norm_weight may be null), and
// every stage reads the normalised copy in the workspace.
// may_fork: the shared expert may run on the library's side stream (not for the entry point that must
// create nothing).
int forward_impl(bool may_fork, bool normed, const void* x_in, const void* norm_weight, float norm_eps,
                 const void* residual, const void* router, const float* router_bias,
                 const void* w_gate, const void* w_up, const void* w_down, const float* s_gate,
                 const float* s_up, const float* s_down, const void* shared_gate,
                 const void* shared_up, const void* shared_down, int32_t T, int32_t D, int32_t E,
                 int32_t K, int32_t F, int32_t F_shared, int32_t tile_m, int32_t act_dtype,
                 int32_t w_dtype, int32_t score_fn, int32_t renormalize, int32_t scale_input,
                 void* workspace, int64_t workspace_bytes, void* out, void* stream) {
  const void* x = x_in;
  const bool act_q = (w_dtype & FS2MOE_ACT_MXFP8) != 0;
  w_dtype &= ~FS2MOE_ACT_MXFP8;
  FS2_REQUIRE(x && router && w_gate && w_up && w_down && out, "forward: null pointer");
  FS2_REQUIRE(T >= 0 && D >= 1 && E >= 1 && K >= 1 && F >= 1 && F_shared >= 0 && tile_m >= 1,
              "forward: bad sizes T=%d D=%d E=%d K=%d F=%d F_shared=%d tile_m=%d", T, D, E, K, F,
              F_shared, tile_m);
  const bool shared = shared_gate || shared_up || shared_down;
  FS2_REQUIRE(!shared || (shared_gate && shared_up && shared_down && F_shared > 0),
              "forward: the shared expert needs its three matrices and F_shared > 0");
  // the raw rows are read by the router only when they are normalised there
  FS2_REQUIRE(normed || x != out, "forward: out must not alias x");
  // the shared expert's output passes through `out` before the residual is read
  FS2_REQUIRE(!(shared && residual == out),
              "forward: with a shared expert out must not alias residual");
  const int64_t need = carve_forward(nullptr, T, D, E, K, F, shared ? F_shared : 0, tile_m,
                                     act_dtype, true, normed).total;
  FS2_REQUIRE(workspace && workspace_bytes >= need,
              "forward: workspace of %lld bytes is smaller than the %lld needed",
              (long long)workspace_bytes, (long long)need);
  FS2_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255u) == 0,
              "forward: workspace must be 256-byte aligned");
  if (T == 0) return FS2MOE_OK;
  // (here for all of its kernels: those of a decode step may be the routed experts' own launches)
  FS2_REQUIRE(!shared || (fs2moe::aligned16(shared_gate) && fs2moe::aligned16(shared_up) &&
                          fs2moe::aligned16(shared_down) && fs2moe::aligned16(out)),
              "forward: the shared expert's matrices and out must be 16-byte aligned");

  // rows are read through the permutation where the expert kernels can (see fs2moe_grouped_swiglu)
  const bool fused = !scale_input && fs2moe::swiglu_gathers_rows(act_dtype, w_dtype, D, F,
                                                                 FS2MOE_MAX_ROWS(T, K, E, tile_m));
  if (act_q) {
    FS2_REQUIRE(w_dtype == FS2MOE_FP8_E4M3 && act_dtype == FS2MOE_BF16 && s_gate && s_up && s_down,
                "forward: FS2MOE_ACT_MXFP8 goes with e4m3 weights, their scales and bf16 rows");
    FS2_REQUIRE(!scale_input, "forward: FS2MOE_ACT_MXFP8 with scale_input is not built into this "
                              "call; use the stage calls");
    FS2_REQUIRE(fs2moe_grouped_swiglu_w8a8_supported(D, F, FS2MOE_MAX_ROWS(T, K, E, tile_m)),
                "forward: FS2MOE_ACT_MXFP8 with D=%d, F=%d: sizes the W8A8 kernels do not take "
                "(fs2moe_grouped_swiglu_w8a8_supported)", D, F);
  }
  // The reference's routing mode multiplies each row by its routing weight on the way in, which
  // dispatch does as it copies the rows.  With at most 16 bf16 tokens (a decode step) the expert
  // kernels stage a few rows in LDS and stream the weights past them: they take the row from x
  // through perm and scale it there, so that no copy is made and dispatch can run inside the router's
  // second kernel as in the other mode.
  const bool scaled_stream = scale_input && !act_q && T <= 16 && D * 2 >= 4 &&
                             fs2moe::swiglu_streams_rows(act_dtype, w_dtype, D, F, E, T);
  const ForwardBuffers b = carve_forward(workspace, T, D, E, K, F, shared ? F_shared : 0, tile_m,
                                         act_dtype, !fused && !act_q && !scaled_stream, normed, act_q,
                                         scaled_stream);
  FS2_REQUIRE(b.total <= need, "forward: internal: the buffers do not fit the workspace");
  // The shared expert's output is the row the routed outputs are added onto (moe.py:143-150).  It depends on the rows
  // only, so it runs beside the routed path where that pays: from the start when it reads the caller's rows, after the
  // router when it reads the rows the router normalises.
  // (forking and joining cost the host four calls, about as long as a whole step of a small layer
  // takes it to launch: D 2048 / F 4096, 16 experts, one token 53 -> 100 us with them, where D 4096 /
  // F 8192 goes 137 -> 129 and Scout's D 5120 / F 8192 173 -> 156; so only where the shared expert
  // streams at least 192 MB of weights)
  const bool big_shared = (int64_t)3 * D * F_shared * fs2moe::elem_size(act_dtype) >= (192ll << 20);
  fs2moe::Branch branch(shared && may_fork && (T <= 16 ? big_shared : fs2moe::branch_pays(T, K, E, D, F, F_shared, act_dtype,
                                                                                          w_dtype, normed, false)), stream);
  const bool beside = branch.beside();
  auto shared_on = [&](void* s, const void* rows) {
    return fs2moe_dense_swiglu(rows, shared_gate, shared_up, shared_down, T, D, F_shared, act_dtype,
                               b.shared_h, out, s);
  };
  auto shared_beside = [&]() -> int {
    if (int rc = branch.fork()) return rc;
    return shared_on(branch.stream(), normed ? b.xn : x_in);
  };
  const int64_t planned = fs2moe::planned_rows((int64_t)T * K, E);
  bool shared_done = false;
  // router, dispatch and the routed experts, with the shared expert forked off on the way
  auto routed_path = [&]() -> int {
    if (!normed)
      if (int rc = branch.mark()) return rc;
    // (with a few tokens and no rows to copy the router's kernel dispatches as well)
    // (and where the experts stream past up to 16 tokens' rows, their first kernel begins with the selection.  Not beside a
    // shared expert: there the selection's own launch costs nothing, D 5120, F 8192, 16 experts, 5 tokens 238.7 us, 239.2)
    fs2moe::Selection later = {};
    const bool selects = !act_q && !beside && fs2moe::swiglu_selects(act_dtype, w_dtype, D, F, E, T);
    fs2moe::DispatchAfterRouter disp = {tile_m,     b.max_rows, b.counts,        b.offsets, b.perm,
                                        b.inv_perm, b.disp_ws,  b.disp_ws_bytes, b.row_w,   selects ? &later : nullptr,
                                        false};
    if (int rc = fs2moe::router_then_dispatch(
            x, normed ? norm_weight : nullptr, normed ? norm_eps : 0.f, normed ? b.xn : nullptr, router,
            router_bias, T, D, E, K, act_dtype, score_fn, renormalize, b.topk_idx, b.topk_w, nullptr,
            b.router_ws, b.router_ws_bytes, b.xe == nullptr ? &disp : nullptr, stream))
      return rc;
    if (normed) x = b.xn;
    // (also where it begins beside the router: in front of the router's launches the four calls of the host's that it takes
    // had a call that the host waits for begin later, 596 tokens, D 1088, F 704, top-6 of 128 143.4 us without a branch, 153.2,
    // now 136.4; 17 such calls 1.00 of the time without, now 0.97, and 0.96 either way as part of a queue)
    if (beside)
      if (int rc = shared_beside()) return rc;
    if (later.partial != nullptr) {
      // (the shared expert's products go into the routed ones' launches)
      const fs2moe::SharedBeside with = {shared_gate, shared_up, shared_down, F_shared, b.shared_h, out};
      shared_done = shared && fs2moe::shared_goes_with_rows(D, F_shared, T);
      return fs2moe::grouped_swiglu_selecting(x, later, w_gate, w_up, w_down, E, D, F, b.max_rows, planned, b.h, b.ye,
                                              shared_done ? &with : nullptr, stream);
    }
    if (!disp.done) {
      if (scaled_stream) {
        if (int rc = fs2moe::dispatch_with_row_weights(b.topk_idx, b.topk_w, T, K, E, tile_m,
                                                       b.max_rows, b.counts, b.offsets, b.perm,
                                                       b.inv_perm, b.row_w, stream))
          return rc;
      } else if (int rc = fs2moe_dispatch(b.topk_idx, b.topk_w, x, T, K, E, D, tile_m, act_dtype,
                                          scale_input, b.max_rows, b.counts, b.offsets, b.perm,
                                          b.inv_perm, b.xe, b.disp_ws, b.disp_ws_bytes, stream)) {
        return rc;
      }
    }
    if (act_q) {
      // the token rows to block-scaled e4m3 once; both products read codes (the first through perm)
      if (int rc = fs2moe_mx_quantize(x, T, D, b.xq, b.xs, stream)) return rc;
      return fs2moe::grouped_swiglu_w8a8_planned(b.xq, b.xs, b.perm, b.counts, b.offsets, w_gate, w_up, w_down,
                                                 s_gate, s_up, s_down, E, D, F, T, b.max_rows, planned, b.hq, b.hs,
                                                 b.ye, stream);
    }
    if (scaled_stream)
      return fs2moe::grouped_swiglu_scaled_rows(x, b.perm, b.row_w, b.counts, b.offsets, w_gate, w_up,
                                                w_down, E, D, F, b.max_rows, planned, b.h, b.ye, T, stream);
    // (a token takes an expert at most once, so no expert has more rows than that)
    return fs2moe::grouped_swiglu_planned(fused ? x : b.xe, fused ? b.perm : nullptr, b.counts, b.offsets,
                                          w_gate, w_up, w_down, s_gate, s_up, s_down, E, D, F, b.max_rows,
                                          planned, act_dtype, w_dtype, b.h, b.ye, T, stream);
  };
  if (int rc = routed_path()) return rc;
  if (int rc = branch.join()) return rc;
  const void* base = nullptr;
  if (shared) {
    if (!beside && !shared_done)
      if (int rc = shared_on(stream, x)) return rc;
    base = out;
  }
  if (residual != nullptr)
    return fs2moe_combine_residual(b.ye, b.inv_perm, b.topk_idx, b.topk_w, base, residual, T, K, D,
                                   act_dtype, scale_input ? 0 : 1, out, stream);
  return fs2moe_combine(b.ye, b.inv_perm, b.topk_idx, b.topk_w, base, T, K, D, act_dtype,
                        scale_input ? 0 : 1, out, stream);
}

}  // namespace

extern "C" int fs2moe_forward(const void* x, const void* residual, const void* router,
                              const float* router_bias,
                              const void* w_gate, const void* w_up, const void* w_down,
                              const float* s_gate, const float* s_up, const float* s_down,
                              const void* shared_gate, const void* shared_up,
                              const void* shared_down, int32_t T, int32_t D, int32_t E, int32_t K,
                              int32_t F, int32_t F_shared, int32_t tile_m, int32_t act_dtype,
                              int32_t w_dtype, int32_t score_fn, int32_t renormalize,
                              int32_t scale_input, void* workspace, int64_t workspace_bytes,
                              void* out, void* stream) {
  return forward_impl(true, false, x, nullptr, 0.f, residual, router, router_bias, w_gate, w_up, w_down,
                      s_gate, s_up, s_down, shared_gate, shared_up, shared_down, T, D, E, K, F,
                      F_shared, tile_m, act_dtype, w_dtype, score_fn, renormalize, scale_input,
                      workspace, workspace_bytes, out, stream);
}

extern "C" int fs2moe_forward_norm(const void* x, const void* norm_weight, float norm_eps,
                                   const void* residual, const void* router,
                                   const float* router_bias,
                                   const void* w_gate, const void* w_up, const void* w_down,
                                   const float* s_gate, const float* s_up, const float* s_down,
                                   const void* shared_gate, const void* shared_up,
                                   const void* shared_down, int32_t T, int32_t D, int32_t E,
                                   int32_t K, int32_t F, int32_t F_shared, int32_t tile_m,
                                   int32_t act_dtype, int32_t w_dtype, int32_t score_fn,
                                   int32_t renormalize, int32_t scale_input, void* workspace,
                                   int64_t workspace_bytes, void* out, void* stream) {
  return forward_impl(true, true, x, norm_weight, norm_eps, residual, router, router_bias, w_gate, w_up,
                      w_down, s_gate, s_up, s_down, shared_gate, shared_up, shared_down, T, D, E, K,
                      F, F_shared, tile_m, act_dtype, w_dtype, score_fn, renormalize, scale_input,
                      workspace, workspace_bytes, out, stream);
}

extern "C" int fs2moe_forward_call(const fs2moe_forward_args* a, void* stream) {
  FS2_REQUIRE(a != nullptr, "forward_call: null pointer");
  return forward_impl(true, a->normed != 0, a->x, a->norm_weight, a->norm_eps, a->residual, a->router,
                      a->router_bias, a->w_gate, a->w_up, a->w_down, a->s_gate, a->s_up, a->s_down,
                      a->shared_gate, a->shared_up, a->shared_down, a->T, a->D, a->E, a->K, a->F, a->F_shared,
                      a->tile_m, a->act_dtype, a->w_dtype, a->score_fn, a->renormalize, a->scale_input,
                      a->workspace, a->workspace_bytes, a->out, stream);
}

// A kernel, where a device-to-device hipMemcpyAsync is a blit kernel between barriers of its own: in
// front of a graph's first kernel 2.3 us instead of 5.4.
namespace {
__global__ __launch_bounds__(256) void copy_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                   int64_t vec, int64_t bytes) {
  const int64_t stride = (int64_t)gridDim.x * 256, first = (int64_t)blockIdx.x * 256 + threadIdx.x;
  for (int64_t i = first; i < vec; i += stride)
    reinterpret_cast<fs2moe::u32x4*>(dst)[i] = reinterpret_cast<const fs2moe::u32x4*>(src)[i];
  for (int64_t i = vec * 16 + first; i < bytes; i += stride) dst[i] = src[i];
}
}  // namespace

extern "C" int fs2moe_copy(const void* src, void* dst, int64_t bytes, void* stream) {
  FS2_REQUIRE(bytes >= 0 && (bytes == 0 || (src && dst)), "copy: bad arguments");
  if (bytes == 0 || src == dst) return FS2MOE_OK;
  const int64_t vec = fs2moe::aligned16(src) && fs2moe::aligned16(dst) ? bytes / 16 : 0;
  const int64_t items = vec > 0 ? vec : bytes, blocks = (items + 255) / 256;
  hipLaunchKernelGGL(copy_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<const uint8_t*>(src),
                     static_cast<uint8_t*>(dst), vec, bytes);
  return fs2moe::check_launch("copy");
}

// ---- the whole layer for callers that cannot allocate ----------------------------------------------
// Every intermediate of fs2moe_forward lives in one array inside the library's own device image, so
// the call needs no workspace from the caller and never touches an allocator.  Every device the
// library runs on holds its own copy of the array, at its own address, until the process ends.
namespace {

static __device__ __align__(256) unsigned char scratch[FS2MOE_STATIC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
// Device address of `scratch` on each device, looked up once per device with that device current.
// Plain word-sized stores of the same value: a race between two first calls is benign.
void* g_scratch_ptr[kMaxDevices] = {};

// The address of this device's copy of the array (the array's name is only a host-side handle and
// must never reach a kernel), or null with the error text set.
void* static_scratch() {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    fs2moe::set_error("forward_static: cannot identify the current device (%s, device %d)",
                      hipGetErrorString(e), dev);
    return nullptr;
  }
  void* p = __atomic_load_n(&g_scratch_ptr[dev], __ATOMIC_ACQUIRE);
  if (p != nullptr) return p;
  e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || p == nullptr) {
    fs2moe::set_error("forward_static: hipGetSymbolAddress failed on device %d: %s", dev,
                      hipGetErrorString(e));
    return nullptr;
  }
  __atomic_store_n(&g_scratch_ptr[dev], p, __ATOMIC_RELEASE);
  return p;
}

}  // namespace

extern "C" int64_t fs2moe_forward_static_capacity(void) { return FS2MOE_STATIC_SCRATCH_BYTES; }

extern "C" int fs2moe_forward_static(const void* x, const void* residual, const void* router,
                                     const float* router_bias, const void* w_gate,
                                     const void* w_up, const void* w_down, const float* s_gate,
                                     const float* s_up, const float* s_down,
                                     const void* shared_gate, const void* shared_up,
                                     const void* shared_down, int32_t T, int32_t D, int32_t E,
                                     int32_t K, int32_t F, int32_t F_shared, int32_t tile_m,
                                     int32_t act_dtype, int32_t w_dtype, int32_t score_fn,
                                     int32_t renormalize, int32_t scale_input, void* out,
                                     void* stream) {
  const int64_t need = fs2moe_forward_workspace_bytes(T, D, E, K, F, F_shared, tile_m, act_dtype);
  FS2_REQUIRE(need >= 0, "forward_static: bad sizes T=%d D=%d E=%d K=%d F=%d F_shared=%d tile_m=%d",
              T, D, E, K, F, F_shared, tile_m);
  FS2_REQUIRE(need <= (int64_t)FS2MOE_STATIC_SCRATCH_BYTES,
              "forward_static: these sizes need %lld bytes of scratch, the built-in array holds "
              "%lld; use fs2moe_forward with a workspace of the caller's",
              (long long)need, (long long)FS2MOE_STATIC_SCRATCH_BYTES);
  void* ws = static_scratch();
  if (ws == nullptr) return FS2MOE_ERR_LAUNCH;
  // Every stage writes what it later reads (nothing in the workspace has to start at zero), so the
  // previous call's contents need no clearing.
  // (everything on the caller's stream: this entry point creates nothing, streams included)
  return forward_impl(false, false, x, nullptr, 0.f, residual, router, router_bias, w_gate, w_up,
                      w_down, s_gate, s_up, s_down, shared_gate, shared_up, shared_down, T, D, E, K,
                      F, F_shared, tile_m, act_dtype, w_dtype, score_fn, renormalize, scale_input, ws,
                      FS2MOE_STATIC_SCRATCH_BYTES, out, stream);
}
