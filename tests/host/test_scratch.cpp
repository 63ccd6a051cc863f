// The library's scratch bookkeeping (csrc/wq_scratch.cpp) on the CPU: the HIP calls it makes are the stand-ins below.
// Prints one line per failed check; exit status 0 when there is none.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <functional>
#include <map>
#include <mutex>
#include <set>
#include <thread>
#include <vector>

#include "wq_scratch.h"

// ---- stand-ins: one device, memory from the host, streams that capture or not
namespace {
std::mutex fake_mu;
size_t live_bytes = 0, peak_bytes = 0;
int mallocs = 0, syncs = 0, failed = 0;
std::map<void*, size_t> sizes;
std::set<hipStream_t> capturing;

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
  *p = malloc(n);  // (untouched pages cost nothing)
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
}

using namespace agq;

namespace {
constexpr size_t MB = (size_t)1 << 20;
hipStream_t stream(int i) { return reinterpret_cast<hipStream_t>((uintptr_t)0x1000 * (i + 1)); }
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
    capturing.insert(hipStreamPerThread);
    expect(stream_scratch(hipStreamPerThread, 1 * MB) == kept, "a warmed stream's buffer under capture");
    expect(stream_scratch(hipStreamPerThread, 64 * MB) == nullptr, "no growth under capture");
    capturing.erase(hipStreamPerThread);
  });
  for (int i = 0; i < 3; ++i)
    in_thread([&] {
      for (size_t b = MB; b <= 8 * MB; b *= 2)
        expect(stream_scratch(hipStreamPerThread, b) != kept, "a captured buffer is not passed on");
    });
  expect(stream_scratch(hipStreamPerThread, 1 * MB) == mine, "and this thread's is still its own");
}
}  // namespace

int main() {
  one_stream_one_buffer();
  per_thread_stream();
  if (!failed) printf("scratch: all checks passed\n");
  return failed ? 1 : 0;
}
