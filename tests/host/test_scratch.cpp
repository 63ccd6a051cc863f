// The library's scratch bookkeeping (csrc/wq_scratch.cpp) on the CPU: the HIP calls it makes are the stand-ins below.
// Prints one line per failed check; exit status 0 when there is none.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <functional>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "wq_scratch.h"

// ---- stand-ins: one device, memory from the host, streams that capture or not
namespace {
std::mutex fake_mu;
size_t live_bytes = 0, peak_bytes = 0;
int mallocs = 0, syncs = 0, failed = 0;
std::map<void*, size_t> sizes;
std::map<hipStream_t, unsigned long long> capturing;  // stream -> capture
unsigned long long captures = 0;

bool any_capture() { return !capturing.empty(); }
void expect(bool ok, const char* what) {
  if (ok) return;
  printf("FAILED: %s\n", what);
  ++failed;
}
}  // namespace

extern "C" {
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) {
  std::lock_guard<std::mutex> l(fake_mu);
  expect(!any_capture(), "a synchronization while a stream captures");
  ++syncs;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> l(fake_mu);
  expect(!any_capture(), "an allocation while a stream captures");
  *p = calloc(1, n);  // (untouched pages cost nothing)
  sizes[*p] = n, live_bytes += n, ++mallocs;
  if (live_bytes > peak_bytes) peak_bytes = live_bytes;
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> l(fake_mu);
  live_bytes -= sizes[p];
  sizes.erase(p);
  free(p);
  return hipSuccess;
}
hipError_t hipMemset(void*, int, size_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
  std::lock_guard<std::mutex> l(fake_mu);
  *st = capturing.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamGetCaptureInfo_v2(hipStream_t s, hipStreamCaptureStatus* st, unsigned long long* id, hipGraph_t*,
                                      const hipGraphNode_t**, size_t*) {
  std::lock_guard<std::mutex> l(fake_mu);
  const auto it = capturing.find(s);
  *st = it != capturing.end() ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  if (it != capturing.end()) *id = it->second;
  return hipSuccess;
}
}

using namespace agq;

namespace {
constexpr size_t MB = (size_t)1 << 20;
hipStream_t stream(int i) { return reinterpret_cast<hipStream_t>((uintptr_t)0x1000 * (i + 1)); }
void begin(hipStream_t s) { capturing[s] = ++captures; }
void end(hipStream_t s) { capturing.erase(s); }
void in_thread(const std::function<void()>& f) { std::thread(f).join(); }

void one_stream_one_buffer() {
  void* const a = stream_scratch(stream(0), 1 * MB);
  expect(a && stream_scratch(stream(0), 4 * MB) == a, "a stream keeps its buffer");
  void* other = nullptr;
  in_thread([&] { other = stream_scratch(stream(0), 1 * MB); });
  expect(other == a, "a stream's buffer is the same in every thread");
  expect(stream_scratch(stream(1), 1 * MB) != a, "two streams have two buffers");
  void* const grown = stream_scratch(stream(0), 5 * MB);
  expect(grown && grown != a && sizes[grown] == 8 * MB && sizes.count(a), "a buffer at least doubles; the old one stays");
}

void per_thread_stream() {
  void* const mine = stream_scratch(hipStreamPerThread, 1 * MB);
  expect(mine && stream_scratch(hipStreamPerThread, 1 * MB) == mine, "a thread keeps its buffer");
  void* theirs = nullptr;
  in_thread([&] { theirs = stream_scratch(hipStreamPerThread, 1 * MB); });
  expect(theirs && theirs != mine, "hipStreamPerThread is another stream, and has another buffer, in another thread");
  // threads that come and go: as many buffers as were alive at once
  const size_t before = live_bytes;
  const int s0 = syncs;
  for (int i = 0; i < 20; ++i)
    in_thread([&] {
      expect(stream_scratch(hipStreamPerThread, 1 * MB) == theirs, "an ended thread's buffer is passed on");
    });
  expect(live_bytes == before && syncs >= s0 + 20, "passed on after a synchronization, without an allocation");
  in_thread([&] {
    expect(stream_scratch(hipStreamPerThread, 1 * MB) == theirs, "passed on");
    expect(stream_scratch(hipStreamPerThread, 6 * MB) != theirs, "grown");
  });
  const size_t grown = live_bytes;
  for (int i = 0; i < 5; ++i)
    in_thread([&] {
      stream_scratch(hipStreamPerThread, 1 * MB);
      stream_scratch(hipStreamPerThread, 6 * MB);
    });
  expect(live_bytes == grown, "what a thread outgrew is passed on too");
  // a buffer that a captured graph addresses stays the graph's
  void* kept = nullptr;
  in_thread([&] {
    kept = stream_scratch(hipStreamPerThread, 1 * MB);
    begin(hipStreamPerThread);
    expect(stream_scratch(hipStreamPerThread, 1 * MB) == kept, "a warmed stream's buffer under capture");
    expect(stream_scratch(hipStreamPerThread, 64 * MB) == nullptr, "no growth under capture");
    end(hipStreamPerThread);
  });
  for (int i = 0; i < 3; ++i)
    in_thread([&] {
      for (size_t b = MB; b <= 8 * MB; b *= 2)
        expect(stream_scratch(hipStreamPerThread, b) != kept, "a captured buffer is not passed on");
    });
  expect(stream_scratch(hipStreamPerThread, 1 * MB) == mine, "and this thread's is still its own");
}

// [counters, end of data) of every piece handed out so far: no two may meet
std::vector<std::pair<uint8_t*, uint8_t*>> taken;
bool apart(const CallScratch& c, size_t bytes) {
  uint8_t *const lo = reinterpret_cast<uint8_t*>(c.cnt), *const hi = c.data + bytes;
  bool ok = c.data >= lo + 4096;
  for (auto& t : taken) ok = ok && (hi <= t.first || t.second <= lo);
  taken.push_back({lo, hi});
  return ok;
}

void captured_calls() {
  begin(stream(7));
  expect(!call_scratch(stream(7), 1 * MB).data, "a capture before any other call has no scratch");
  end(stream(7));
  const CallScratch eager = call_scratch(stream(8), 1 * MB);
  expect(eager.data && eager.data == reinterpret_cast<uint8_t*>(eager.cnt) + 4096, "a call's scratch: counters, data");
  expect(static_cast<void*>(eager.cnt) == stream_scratch(stream(8), 1 * MB), "outside a capture: the stream's");
  expect(apart(eager, 1 * MB), "first");
  const size_t before = live_bytes;
  // from the warmed stream and from one that the library has not seen, one after the other and at once
  for (int round = 0; round < 2; ++round) {
    begin(stream(8));
    begin(stream(9));
    const CallScratch a = call_scratch(stream(8), 1 * MB), b = call_scratch(stream(9), 2 * MB);
    expect(a.data && b.data && apart(a, 1 * MB) && apart(b, 2 * MB), "a captured call shares with nothing else");
    expect(call_scratch(stream(8), 1 * MB).data == a.data && call_scratch(stream(9), 1 * MB).data == b.data,
           "the calls of one capture on one stream share");
    const CallScratch more = call_scratch(stream(8), 5 * MB);
    expect(more.data && apart(more, 5 * MB), "a larger call of a capture gets a larger piece");
    expect(call_scratch(stream(8), 1 * MB).data == more.data, "which the later ones share");
    end(stream(8));
    end(stream(9));
    expect(call_scratch(stream(8), 1 * MB).data == eager.data, "calls outside a capture keep the stream's");
  }
  begin(stream(8));
  begin(hipStreamPerThread);
  CallScratch here = call_scratch(hipStreamPerThread, 1 * MB), there;
  in_thread([&] { there = call_scratch(hipStreamPerThread, 1 * MB); });
  expect(apart(here, 1 * MB) && apart(there, 1 * MB), "hipStreamPerThread: by thread");
  end(hipStreamPerThread);
  // the fixed buffer of the entry point that allocates nothing comes first
  static uint8_t fixed[64 << 10];
  scratch_override() = {fixed, sizeof(fixed), true};
  expect(static_cast<void*>(call_scratch(stream(8), 60 << 10).cnt) == fixed, "the fixed buffer");
  expect(!call_scratch(stream(8), 64 << 10).data, "which is too small for 64 KB beside the counters");
  scratch_override() = ScratchOverride();
  end(stream(8));
  // the reserve ends; then there is none, and nothing new was allocated
  int got = 0;
  for (int i = 0; i < 400; ++i) {
    begin(stream(11));
    const CallScratch c = call_scratch(stream(11), 1 * MB);
    if (c.data) expect(apart(c, 1 * MB), "pieces are apart to the end"), ++got;
    end(stream(11));
  }
  expect(got > 200 && got < 256, "256 MB in all");
  expect(live_bytes <= before + 4 * MB + 8 * MB, "captured calls allocate nothing");
}
}  // namespace

int main() {
  one_stream_one_buffer();
  per_thread_stream();
  captured_calls();
  if (!failed) printf("scratch: all checks passed\n");
  return failed ? 1 : 0;
}
