// common.hpp -- error reporting and per-stream workspace for the sts_attn library.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <mutex>
#include <string>

#include "sts_attn.h"

namespace sts {

// Records `msg` as the calling thread's last error and returns `code`.
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
// Clears the calling thread's last error.
void clear_error();
const char* last_error_cstr();

#define STS_HIP(call)                                                              \
  do {                                                                             \
    hipError_t e_ = (call);                                                        \
    if (e_ != hipSuccess)                                                          \
      return ::sts::fail(STS_ERR_HIP, "%s failed: %s (%d) at %s:%d", #call,        \
                         hipGetErrorString(e_), (int)e_, __FILE__, __LINE__);      \
  } while (0)

#define STS_CHECK(cond, ...)                                                       \
  do {                                                                             \
    if (!(cond)) return ::sts::fail(STS_ERR_INVALID, __VA_ARGS__);                 \
  } while (0)

// Split-KV partial results and arrival counters for one (device, stream).
struct Workspace {
  float* part = nullptr;       // partial (acc[D], m, l) records
  size_t part_floats = 0;
  uint32_t* counters = nullptr;  // one arrival counter per (stream, head); zero between calls
  size_t n_counters = 0;
};

// Returns a workspace for `stream` on the current device holding at least the
// requested sizes.  Growing allocates new buffers (new counters zero-filled on
// the stream) and retires the old ones without freeing them, so work queued
// earlier and graphs captured earlier stay valid.  Fails with STS_ERR_STATE
// when it would have to allocate while the stream is being captured.
int get_workspace(hipStream_t stream, size_t part_floats, size_t n_counters, Workspace** out);

// get_workspace for callers that have another way: *out stays null, with
// STS_OK, where the workspace would have to grow and cannot (`stream` is being
// captured, memory is short).  The allocation is made in relaxed capture mode,
// so that it does not break a capture of another stream in progress.
int try_workspace(hipStream_t stream, size_t part_floats, size_t n_counters, Workspace** out);

// Memory through which the launches of one call hand data to one another, per
// (device, stream) and apart from Workspace.  Its holder has it alone until it
// goes out of scope, which it does once the call's last launch is enqueued:
// calls of other host threads on the same stream wait for that, so that their
// launches come after all of this call's and not between two of them.
// part is null where the caller has to take its way without: while `stream` is
// being captured, so that a graph shares no memory with another one or with
// eager calls beside its replays and its result does not depend on what ran
// before the capture, and where memory is short.  Growing happens in relaxed
// capture mode, so that it does not break a capture of another stream in
// progress, and retires the old buffers as Workspace does.
class Scratch {
 public:
  Scratch(hipStream_t stream, size_t part_floats, size_t n_counters);
  Scratch(const Scratch&) = delete;
  Scratch& operator=(const Scratch&) = delete;
  float* part = nullptr;
  uint32_t* counters = nullptr;  // zero between calls

 private:
  std::unique_lock<std::mutex> held_;
};

// Number of compute units of the current device (cached per device).
int device_cu_count();

// Poll bound of the kernels' bounded waits (0 restores the default, 2^24).
void set_wait_limit(uint32_t polls);
uint32_t wait_limit();

}  // namespace sts
