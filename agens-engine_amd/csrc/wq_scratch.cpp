// Library scratch per (device, stream), as the reference keeps its split-K partials and counters
// (w4_gemv.cu:2096-2118): allocated zero-filled on first use and grown (at least doubling) when a launch needs more,
// never inside a stream capture (null then: the caller takes a path without scratch).  Every buffer handed out is held
// until the process ends, the replaced ones included, so launches still in flight and graphs captured before a growth
// keep valid memory.  Launches on one stream are ordered, so they share it safely.  Users keep their counters (the
// first 4 KB) at zero between launches.
//
// hipStreamPerThread is one handle for a stream of its own in every host thread: its scratch is per thread.  When a
// thread ends, its buffer goes to the next thread that asks for no more (after a device synchronization), so that a
// program whose threads come and go holds as many as were alive at once; a buffer that a captured graph addresses is
// not passed on.
//
// A caller that must not allocate (ak_wq_gemv_kt_multi_noalloc) installs a fixed buffer for the calling thread first:
// then stream_scratch returns that buffer when it is large enough and null otherwise, and never allocates.
#include "wq_scratch.h"

#include <stdint.h>

#include <atomic>
#include <map>
#include <tuple>
#include <utility>
#include <vector>

namespace agq {
namespace {

struct Buf {
  void* p = nullptr;
  size_t bytes = 0;
  bool captured = false;  // handed out under a stream capture
};

struct Pool {
  std::mutex mu;
  std::map<std::tuple<int, hipStream_t, uint64_t>, Buf> bufs;  // (device, stream, thread_of(stream))
  std::vector<std::pair<int, Buf>> idle;                       // (device, buffer) of threads that ended
};

Pool& pool() {
  static Pool* const p = new Pool;  // never destroyed: threads may end after main returns
  return *p;
}

struct ThreadId {
  const uint64_t id;
  ThreadId() : id(next()) {}
  ~ThreadId() {
    Pool& P = pool();
    std::lock_guard<std::mutex> lock(P.mu);
    for (auto it = P.bufs.begin(); it != P.bufs.end();) {
      if (std::get<2>(it->first) != id) {
        ++it;
        continue;
      }
      if (it->second.p && !it->second.captured) P.idle.push_back({std::get<0>(it->first), it->second});
      it = P.bufs.erase(it);
    }
  }
  static uint64_t next() {
    static std::atomic<uint64_t> n{0};
    return ++n;  // never reused
  }
};

uint64_t thread_of(hipStream_t s) {
  if (s != hipStreamPerThread) return 0;
  static thread_local ThreadId t;
  return t.id;
}

}  // namespace

ScratchOverride& scratch_override() {
  static thread_local ScratchOverride o;
  return o;
}

std::mutex& scratch_mutex(hipStream_t s) {
  static std::mutex m[64];  // streams share one only by chance of their address
  return m[(reinterpret_cast<uintptr_t>(s) >> 6) & 63];
}

void* stream_scratch(hipStream_t s, size_t bytes) {
  const ScratchOverride& o = scratch_override();
  if (o.on) return bytes <= o.bytes ? o.p : nullptr;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  const uint64_t thread = thread_of(s);
  Pool& P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  Buf& b = P.bufs[{dev, s, thread}];
  const bool have = b.p && b.bytes >= bytes;
  if (have && (!thread || b.captured)) return b.p;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  const bool ok = hipStreamIsCapturing(s, &cs) == hipSuccess;
  if (!ok || cs != hipStreamCaptureStatusNone) {
    if (!ok) (void)hipGetLastError();
    if (!have) return nullptr;
    b.captured = true;
    return b.p;
  }
  if (have) return b.p;
  // a per-thread stream gives the buffer that it outgrows back as well
  auto replace_with = [&](Buf n) {
    if (thread && b.p && !b.captured) P.idle.push_back({dev, b});
    b = n;
    return b.p;
  };
  for (size_t i = 0; thread && i < P.idle.size(); ++i)
    if (P.idle[i].first == dev && P.idle[i].second.bytes >= bytes) {
      if (hipDeviceSynchronize() != hipSuccess) {  // the last launches in it
        (void)hipGetLastError();
        return nullptr;
      }
      const Buf n = P.idle[i].second;
      P.idle.erase(P.idle.begin() + (long)i);
      return replace_with(n);
    }
  // at least double: a replaced buffer is kept, not freed (a graph captured before the growth still addresses it), so
  // the replaced buffers stay below the current one in total
  size_t want = bytes > ((size_t)4 << 20) ? bytes : ((size_t)4 << 20);
  if (b.p && want < 2 * b.bytes) want = 2 * b.bytes;
  void* p = nullptr;
  if (hipMalloc(&p, want) != hipSuccess || hipMemset(p, 0, want) != hipSuccess || hipDeviceSynchronize() != hipSuccess) {
    if (p) (void)hipFree(p);
    (void)hipGetLastError();
    return nullptr;
  }
  return replace_with({p, want, false});
}

}  // namespace agq
