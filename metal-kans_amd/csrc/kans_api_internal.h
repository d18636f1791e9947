// Internal declarations shared by the runtime and kernel translation units.
#pragma once
#include <hip/hip_runtime.h>
#include "kans_common.h"
#include "../../include/kans_hip.h"
#include <memory>
#include <mutex>
#include <vector>

namespace kans {

// One fused dense launch (see kans_dense.hip).
struct DenseLaunch {
  int dtype, basis, has_base;
  int x_dtype, y_dtype;  // element types of X and Y: dtype, or DT_F32
  const void* X; long ldx;
  const void* Wt; int nob_pad;
  const float* bias;    // [D_out] constant term per output (bias, folded T_0 coefficients) or null
  void* Y; long ldy;
  float* part;          // split workspace (splits * B * D_out floats) or null
  int B, D_in, D_out, nfb;
  BasisParams bp;
  int wm, nb, splits;   // tile config
  int ks = 1;           // wave groups per workgroup (4-wave block kernel, block_wave_groups_ok)
  int pair = 1;         // block kernels: two feature blocks per LDS stage when they fit (kan_fused_block)
};

// A layer's weights on the device into the fused kernels' layout (kans_dense.hip): W / Wb / bias of
// src_dtype (the layer dtype, or DT_F32 for a converting upload; Wb / bias may be null) into Wt and, when
// bias_out is set, the constant term per output.
struct WeightUpload {
  int src_dtype, dtype;
  const void *W, *Wb, *bias;
  void* Wt;
  float* bias_out;
  int D_in, D_out, K, has_base;
  int sparse;           // layout of kan_fused_split_sparse (fp32 B-spline)
  int fold;             // T_0 coefficients go into bias_out (BasisParams::k0)
  int nfb, nob_pad;
};

// RBF parameters (centres, scaled centres, recurrence eligibility) of bp (bp.K set) from K centres and
// inv_denominator = 1/(2h^2); false (bp unchanged) when inv_den is negative or not finite
// (kans_runtime.hip).
bool kans_set_rbf_params(BasisParams& bp, const float* centers, float inv_den);

// Host <-> device staging through pinned memory, the host copies split over worker threads and
// overlapped with the DMAs (kans_staging.hip; call with the library lock held).
// stage_in: `rows` rows of `row_bytes` bytes, contiguous in host src, into device rows of `pitch` bytes
// (the tail of each row zeroed) through the pinned buffer `pin` (>= rows * pitch bytes).  Returns once
// every DMA is enqueued on st; `pin` stays in use until st has passed them.
int stage_in(void* dst, const void* src, size_t row_bytes, size_t pitch, long rows, void* pin, hipStream_t st);
// stage_out: `bytes` from device src, after the work already on st, into host dst through the pinned
// buffer `pin` (>= bytes).  Returns when dst holds them.
int stage_out(void* dst, const void* src, size_t bytes, void* pin, hipStream_t st);
// The same in two parts, for transfers from several streams: stage_out_enqueue adds the device -> pinned
// copies of one range (after the work already on st) to `out`; stage_out_drain waits for the pieces in
// the order they were added and copies each into host memory as it lands.
struct StagedOut {
  struct Piece {
    char* dst;
    const char* pin;
    size_t bytes;
  };
  std::vector<Piece> pieces;
  size_t bytes = 0;
};
int stage_out_enqueue(StagedOut& out, void* dst, const void* src, size_t bytes, void* pin, hipStream_t st);
int stage_out_drain(StagedOut& out);

}  // namespace kans

int kans_fail(int code, const char* fmt, ...);
#define HIP_TRY(expr)                                                                       \
  do {                                                                                      \
    hipError_t _e = (expr);                                                                 \
    if (_e != hipSuccess)                                                                   \
      return kans_fail(KANS_ERR_HIP, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(_e), \
                       __FILE__, __LINE__);                                                 \
  } while (0)

// Grow-only device buffer.
struct DevBuf {
  void* p = nullptr;
  size_t cap = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() { if (p) (void)hipFree(p); }
  int reserve(size_t bytes) {
    if (bytes <= cap) return 0;
    if (p) HIP_TRY(hipFree(p));
    p = nullptr;
    cap = 0;
    HIP_TRY(hipMalloc(&p, bytes));
    cap = bytes;
    return 0;
  }
};

// Per-device set-up of kans_gated_forward_noalloc's scratch (kans_qruntime.hip);
// called by the library's initialisation with `device` current.
int kans_noalloc_setup(int device);
hipStream_t kans_default_stream();
// The stream of an entry point's `stream` argument: NULL is the library's own, KANS_STREAM_LEGACY the HIP
// default stream (whose handle is itself null; the runtime's own pseudo-handle for it must not reach event
// calls: waiting for an event recorded through it crashed).
inline hipStream_t kans_caller_stream(void* stream) {
  if (!stream) return kans_default_stream();
  return stream == KANS_STREAM_LEGACY ? (hipStream_t) nullptr : (hipStream_t)stream;
}
// Whether st is under graph capture (the default stream never is).
hipError_t kans_capturing(hipStream_t st, bool* capturing);
// Workspace for the partial sums of a split kernel on stream st, `bytes` large: one per stream, which all
// calls on the stream share, since their kernels run one after the other (library lock held; st not under
// capture by a caller).  Null where there is none -- no memory for it, or hipStreamPerThread, one handle
// for several streams: the caller then runs unsplit.  It grows with the calls and stays until the next
// larger request or until kMaxWorkspaces other streams have asked since; the library's last object frees all
// but a few MB (WorkspaceUser).
float* kans_stream_workspace(hipStream_t st, size_t bytes);
struct WorkspaceUser {
  WorkspaceUser();
  ~WorkspaceUser();
  WorkspaceUser(const WorkspaceUser&) = delete;
  WorkspaceUser& operator=(const WorkspaceUser&) = delete;
};
// Allows this thread the calls that a capture running in another one forbids by default (waiting for the
// device or an event, allocations); none of them concerns a capturing stream.
struct CaptureRelaxed {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  CaptureRelaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~CaptureRelaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};
// Workspaces of calls that callers have captured on an object's behalf.  A graph keeps the pointer and may be
// replayed beside any other work, so each call has its own, until the object is destroyed (as its weights are,
// which the graph holds too).  Null once they hold kMaxCapturedBytes, or without memory.
struct CapturedWorkspaces {
  std::vector<std::unique_ptr<DevBuf>> bufs;
  size_t bytes = 0;
  float* take(size_t n);
};
constexpr size_t kMaxCapturedBytes = size_t(256) << 20;
// The workspace of a split call on st: the stream's, or one of its own under a caller's capture.
// *part is null where there is none.
int kans_split_workspace(CapturedWorkspaces& captured, hipStream_t st, size_t bytes, float** part);
// fp32 Chebyshev forward (no base branch) of host X on device-resident fp32 weights (kans_runtime.hip);
// call with the library lock held.
int kans_ref_cheby_forward_devw_locked(const float* X, const float* W_dev, const float* bias_dev, float* Y, int B,
                                       int D_in, int D_out, int K, int has_bias);

// Library lock (serialises every entry point that touches device state), lazy
// device initialisation (call with the lock held) and the grow-only pinned
// staging buffers of the synchronous host-pointer entry points (which = 0 in,
// 1 out; lock held).
std::mutex& kans_mutex();
int kans_ensure_init();
int kans_pinned_stage(int which, size_t bytes, void** p);

// Grow-only pinned host buffer.
struct Pinned {
  void* p = nullptr;
  size_t cap = 0;
};
inline int pinned_reserve(Pinned& b, size_t bytes) {
  if (bytes <= b.cap) return 0;
  if (b.p) HIP_TRY(hipHostFree(b.p));
  b.p = nullptr;
  b.cap = 0;
  size_t cap = bytes + bytes / 4;
  HIP_TRY(hipHostMalloc(&b.p, cap, hipHostMallocDefault));
  b.cap = cap;
  return 0;
}
