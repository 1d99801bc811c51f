// Shared host-side plumbing of the gfx950 library: error reporting, per-device workspace,
// stream synchronisation flag.  Device helpers live in f3d_device.h.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include "../../include/f3d_hip.h"

namespace f3d {

// Message of the last failing call on this thread (returned by f3d_last_error()).
void set_error(const char* fmt, ...) __attribute__((format(printf, 1, 2)));

// Grow-only scratch buffer owned by the library, one per device.  Work that uses it is ordered on
// the caller's stream; calls that overlap on different streams of one device must not share it, so
// every entry point that needs scratch documents that it is not re-entrant per device.
// `stream`: the caller's stream; when the buffer has to grow while that stream is being captured the call fails with a
// message (warm the shapes up outside capture) and does not touch the device.
// Returns nullptr (and sets the error) on failure.
void* workspace(int device, size_t bytes, hipStream_t stream);

// Device memory for the weights a dense op prepares per call (LayerNorm folded into the weight, fragment-major
// copies): the buffer the caller staged with f3d_stage_weights for this call, else the per-device workspace.
// *ready: the staged buffer already holds this call's prepared weights, the preparation launch is skipped.
// nullptr + error message when the staged buffer is too small or the workspace cannot grow.
void* weight_area(int device, size_t bytes, bool* ready, hipStream_t stream);
// Declared at the top of every dense entry point: whatever the call does, the staging ends with it.  An entry point that
// asks for a weight_area returns succeeded() (F3D_OK) behind its last launch: f3d_staged_weights_kept then says so.
struct StagedWeightsScope {
  int succeeded();
  ~StagedWeightsScope();
};

// This device's copy of the fixed scratch array behind f3d_batch_psh_scatter_pad_hash_noalloc (resolved on the first
// call per device; f3d_init_dev_info does it ahead of time).  nullptr + error message on failure.
uint32_t* psh_noalloc_scratch(int device);

bool sync_stream_enabled();
uint32_t global_seed();
int rebalance_mode();
// 0x80000000 when the voxel quantiser divides (f3d_set_quantiser(1)), else 0: OR-ed into a kernel's num_vox argument
uint32_t quantiser_bit();

#define F3D_CHECK_ARG(cond, ...)            \
  do {                                      \
    if (!(cond)) {                          \
      ::f3d::set_error(__VA_ARGS__);        \
      return F3D_ERR_INVALID;               \
    }                                       \
  } while (0)

#define F3D_CHECK_HIP(expr)                                                              \
  do {                                                                                   \
    hipError_t _e = (expr);                                                              \
    if (_e != hipSuccess) {                                                              \
      ::f3d::set_error("HIP error %d (%s) at %s:%d", (int)_e, hipGetErrorString(_e),    \
                       __FILE__, __LINE__);                                              \
      return F3D_ERR_RUNTIME;                                                            \
    }                                                                                    \
  } while (0)

// RAII bracket reproducing the reference's optional stream synchronisation around an op
// (src/psh/batch_psh_bucket_dispatcher.cu:278-280, 323-325).
// A stream that is being captured is left alone (synchronising it would invalidate the capture).
struct SyncBracket {
  hipStream_t s;
  bool on;
  explicit SyncBracket(hipStream_t stream) : s(stream), on(false) {
    if (!sync_stream_enabled()) return;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    on = hipStreamIsCapturing(s, &st) == hipSuccess && st == hipStreamCaptureStatusNone;
    if (on) (void)hipStreamSynchronize(s);
  }
  ~SyncBracket() {
    if (on) (void)hipStreamSynchronize(s);
  }
};

// Makes `device` current for the lifetime of the object and restores the previous one.
struct DeviceGuard {
  int prev = -1;
  bool ok = true;
  explicit DeviceGuard(int device) {
    if (hipGetDevice(&prev) != hipSuccess) prev = -1;
    if (prev != device) ok = hipSetDevice(device) == hipSuccess;
  }
  ~DeviceGuard() {
    int cur = -1;
    if (prev >= 0 && hipGetDevice(&cur) == hipSuccess && cur != prev) (void)hipSetDevice(prev);
  }
};

static inline uint32_t cdiv_u32(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

// Whether y [rows][cols_y] may share an element with x [rows][cols_x] (row strides in elements).  Matrices whose address
// ranges meet are told apart only when their rows have one pitch: y may then be other columns of the same buffer.
static inline bool rows_overlap(const void* x, uint32_t ldx, uint32_t cols_x, const void* y, uint32_t ldy, uint32_t cols_y,
                                uint32_t rows) {
  if (rows == 0 || cols_x == 0 || cols_y == 0) return false;
  const uint64_t x0 = (uintptr_t)x / 2, y0 = (uintptr_t)y / 2;      // in elements of two bytes
  if (x0 + (uint64_t)(rows - 1) * ldx + cols_x <= y0 || y0 + (uint64_t)(rows - 1) * ldy + cols_y <= x0) return false;
  if (ldx != ldy) return true;
  const uint64_t at = y0 >= x0 ? (y0 - x0) % ldx : (ldx - (x0 - y0) % ldx) % ldx;   // y's first column in a row of x
  return at < cols_x || at + cols_y > ldx;
}

}  // namespace f3d
