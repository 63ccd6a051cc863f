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
// Captured calls.  A graph runs whenever and wherever it is launched: beside other graphs captured from the same stream,
// and beside later calls on it.  The calls of one capture on one stream therefore share a piece of a reserve (call_scratch)
// that nothing else uses.  The reserve is 256 MB per device, allocated with the first call outside a capture that needs
// scratch, on whatever stream; a piece is what the largest of its calls needs (a 16-token decode step of 27648 inputs 3
// MB, 64 tokens 16 MB).  Pieces are not given back: an executable graph updated from another one (hipGraphExecUpdate) goes
// on addressing the other's pieces after that one is destroyed, and the runtime does not tell.  When the reserve is used
// up, calls are captured in the form without scratch.  (The split-K launches of the small-M kernels work in stream_scratch
// under a capture as well, as the reference's do: graphs with such launches captured from one stream run in order.)
//
// A caller that must not allocate (ak_wq_gemv_kt_multi_noalloc) installs a fixed buffer for the calling thread first:
// then both functions return that buffer when it is large enough and null otherwise, and never allocate.
#include "wq_scratch.h"

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

constexpr size_t kCounters = 4096, kReserve = (size_t)256 << 20;
struct Reserve {
  uint8_t* p = nullptr;
  size_t used = 0;
  bool tried = false;
};

struct Pool {
  std::mutex mu;
  std::map<std::tuple<int, hipStream_t, uint64_t>, Buf> bufs;  // (device, stream, thread_of(stream))
  std::vector<std::pair<int, Buf>> idle;                       // (device, buffer) of threads that ended
  std::map<int, Reserve> reserve;                              // by device
  // (device, stream, thread_of(stream), capture) -> the piece its calls share
  std::map<std::tuple<int, hipStream_t, uint64_t, unsigned long long>, Buf> pieces;
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
  // at least double, up to the most that a call asks for: a replaced buffer is kept, not freed (a graph captured before
  // the growth still addresses it), so the replaced buffers stay below twice the current one in total
  size_t want = bytes > ((size_t)4 << 20) ? bytes : ((size_t)4 << 20);
  const size_t twice = 2 * b.bytes < kMaxCallScratch + kCounters ? 2 * b.bytes : kMaxCallScratch + kCounters;
  if (b.p && want < twice) want = twice;
  void* p = nullptr;
  if (hipMalloc(&p, want) != hipSuccess || hipMemset(p, 0, want) != hipSuccess || hipDeviceSynchronize() != hipSuccess) {
    if (p) (void)hipFree(p);
    (void)hipGetLastError();
    return nullptr;
  }
  return replace_with({p, want, false});
}

CallScratch call_scratch(hipStream_t s, size_t bytes) {
  CallScratch c;
  auto in = [&](void* p) {
    if (p) c.cnt = static_cast<int*>(p), c.data = static_cast<uint8_t*>(p) + kCounters;
    return c;
  };
  bytes += kCounters;
  if (scratch_override().on) return in(stream_scratch(s, bytes));
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  // (the legacy stream is never captured, and may not be asked while another one is)
  if (s && s != hipStreamLegacy && hipStreamGetCaptureInfo_v2(s, &cs, &id, nullptr, nullptr, nullptr) != hipSuccess) {
    (void)hipGetLastError();
    return c;
  }
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return c;
  Pool& P = pool();
  if (cs == hipStreamCaptureStatusNone) {
    void* const z = stream_scratch(s, bytes);
    std::lock_guard<std::mutex> lock(P.mu);
    Reserve& r = P.reserve[dev];
    if (z && !r.tried) {
      r.tried = true;
      void* p = nullptr;
      if (hipMalloc(&p, kReserve) == hipSuccess && hipMemset(p, 0, kReserve) == hipSuccess &&
          hipDeviceSynchronize() == hipSuccess) {
        r.p = static_cast<uint8_t*>(p);
      } else {
        if (p) (void)hipFree(p);
        (void)hipGetLastError();
      }
    }
    return in(z);
  }
  if (cs != hipStreamCaptureStatusActive) return c;
  const uint64_t thread = thread_of(s);
  std::lock_guard<std::mutex> lock(P.mu);
  const std::tuple<int, hipStream_t, uint64_t, unsigned long long> key{dev, s, thread, id};
  const auto it = P.pieces.find(key);
  if (it != P.pieces.end() && it->second.bytes >= bytes) return in(it->second.p);
  Reserve& r = P.reserve[dev];
  bytes = (bytes + 4095) & ~(size_t)4095;
  if (!r.p || kReserve - r.used < bytes) return c;
  void* const p = r.p + r.used;
  r.used += bytes;
  P.pieces[key] = {p, bytes, true};  // (a smaller piece of the capture stays with its earlier calls)
  return in(p);
}

}  // namespace agq
