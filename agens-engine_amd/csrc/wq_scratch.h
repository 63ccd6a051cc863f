// Library scratch of the launches whose kernels hand data to each other or to other workgroups.  Host code only.
#pragma once
#include <hip/hip_runtime_api.h>
#include <stddef.h>
#include <stdint.h>

#include <mutex>

namespace agq {

// A fixed scratch buffer that replaces the per-stream library scratch for the calling host thread while `on` (the
// entry point that allocates nothing installs it around its launches).
struct ScratchOverride {
  void* p = nullptr;
  size_t bytes = 0;
  bool on = false;
};
ScratchOverride& scratch_override();

// Held while a call on stream s enqueues kernels that work in the stream's scratch: calls of two host threads on one
// stream are then ordered as wholes, also those whose kernels hand data to each other through the scratch.
std::mutex& scratch_mutex(hipStream_t s);

// The scratch of stream s on the current device, at least `bytes` long; null without it (see wq_scratch.cpp).
void* stream_scratch(hipStream_t s, size_t bytes);

// The most data that one call asks of call_scratch: the launch shapes that need more are not considered
constexpr size_t kMaxCallScratch = (size_t)256 << 20;

// The same for a call that may be captured: 4 KB of counters (zero between launches) and `bytes` of data that no other
// stream and no other graph works in; null pointers without it.
struct CallScratch {
  int* cnt = nullptr;
  uint8_t* data = nullptr;
};
CallScratch call_scratch(hipStream_t s, size_t bytes);

}  // namespace agq
