// Internal helpers shared by the runtime and the attention kernels.
// Host-side error reporting, the library stream and the workspace cache.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "../../include/tt_attn.h"

namespace tt {

// Records a message for tt_last_error() and returns `code`.
int fail(int code, const std::string& msg);
// Clears the last error and returns TT_OK.
int ok();
// Maps a HIP status to TT_ERR_HIP with the call site.
int hip_fail(hipError_t e, const char* what);

// The library stream (created by tt_init on first use).
hipStream_t stream_or_default(void* s);
int ensure_init();
// Compute units of the bound device (after ensure_init).
int device_cu_count();

// Records the next instrumentation event (tt_set_launch_events) after a
// kernel launch on `s`; a no-op unless instrumentation is enabled.
void after_launch(hipStream_t s);

// Whether `s` is being captured into a graph (then a launcher allocates
// nothing and leaves no scratch address behind).
bool stream_capturing(hipStream_t s);

// Whether [p, p + bytes) lies inside one block that tt_malloc or
// tt_malloc_ordered handed out and that was not freed.
bool device_block_holds(const void* p, size_t bytes);

// The allocation-free backward's scratch: a static device array of
// kNoAllocScratchBytes whose device address tt_init looks up once per
// device.  Returns nullptr before tt_init; *bytes gets the array's size.
constexpr size_t kNoAllocScratchBytes = size_t(16) << 20;
void* noalloc_scratch(size_t* bytes);

// Device scratch of the attention launchers: one buffer per (stream, user),
// grown on demand and kept for reuse.  A lease holds the workspace lock from
// get() until it is destroyed: keep it alive until every kernel that reads
// the buffer has been launched on that stream.  A user that also runs under
// capture (the fp32 forward, the backward, the long decode splits) shares its
// buffer with no other: their requests would replace the one a graph keeps.
enum { kWsBackwardRows = 0, kWsDecodePartials = 1, kWsForwardSplits = 2, kWsSoftmaxPartials = 3, kWsGemmSplits = 4, kWsDecodeShort = 5, kWsForwardSplitsBf16 = 6 };
class WorkspaceLease {
 public:
  WorkspaceLease();
  ~WorkspaceLease();
  WorkspaceLease(const WorkspaceLease&) = delete;
  WorkspaceLease& operator=(const WorkspaceLease&) = delete;
  // *uses (optional): earlier get() calls that returned the same buffer (0:
  // a new buffer with undefined contents).
  int get(hipStream_t stream, int user, size_t bytes, void** ptr, uint64_t* uses = nullptr);
  // For a launcher that also runs without the buffer: true and *ptr, or false
  // where none may be had (a refused allocation; a stream under capture, whose
  // graph would keep the address; the library stream under capture, which a new
  // buffer would order the stream behind).  Leaves captures of other streams
  // alone: an allocation of this thread would end them otherwise.
  bool get_optional(hipStream_t stream, int user, size_t bytes, void** ptr, uint64_t* uses = nullptr);
  // The same for a user whose requests are all of one size: its buffer is never
  // replaced, so a graph may keep the address, and a stream under capture gets
  // the one that an earlier call left.
  bool get_fixed(hipStream_t stream, int user, size_t bytes, void** ptr);

 private:
  struct Impl;
  Impl* impl_;
};

}  // namespace tt

#define TT_HIP(call)                                   \
  do {                                                 \
    hipError_t e_ = (call);                            \
    if (e_ != hipSuccess) return tt::hip_fail(e_, #call); \
  } while (0)

#define TT_LAUNCH_CHECK(what)                                  \
  do {                                                         \
    hipError_t e_ = hipGetLastError();                         \
    if (e_ != hipSuccess) return tt::hip_fail(e_, what);       \
  } while (0)

namespace tt {
// A one-dimensional launch holds at most 2^32 - 1 work-items (the dispatch
// packet counts the grid in work-items, not workgroups).
inline bool grid_fits(int64_t workgroups, int64_t threads) {
  return workgroups >= 0 && workgroups <= int64_t(0xffffffffu) / threads;
}
}  // namespace tt

// Launch-error check plus the instrumentation hook, for kernels on stream s.
#define TT_LAUNCHED(what, s)    \
  do {                          \
    TT_LAUNCH_CHECK(what);      \
    tt::after_launch(s);        \
  } while (0)
