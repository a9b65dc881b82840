// A host stand-in for the HIP calls that the library's host code makes around copies and
// waits: streams that run their work in order on a thread of their own, late, so that code
// which does not wait for an event or a stream reads what is not there yet.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <thread>

namespace fake {

inline bool refuse_pinned = false;
inline std::atomic<int> pinned_allocations{0}, pinned_alive{0}, copies{0};
inline std::atomic<int> stream_status{-1};  // what a query answers; -1: by the stream's work

struct Stream {
  std::mutex mu;
  std::condition_variable cv;
  std::deque<std::function<void()>> work;
  long queued = 0, done = 0;
  bool stop = false;
  std::thread thread{[this] { loop(); }};
  ~Stream() {
    {
      std::lock_guard<std::mutex> lock(mu);
      stop = true;
    }
    cv.notify_all();
    thread.join();
  }
  void loop() {
    std::unique_lock<std::mutex> lock(mu);
    for (;;) {
      cv.wait(lock, [&] { return stop || !work.empty(); });
      if (work.empty()) return;
      auto f = std::move(work.front());
      work.pop_front();
      lock.unlock();
      std::this_thread::sleep_for(std::chrono::microseconds(50));
      f();
      lock.lock();
      ++done;
      cv.notify_all();
    }
  }
  long put(std::function<void()> f) {
    std::lock_guard<std::mutex> lock(mu);
    work.push_back(std::move(f));
    cv.notify_all();
    return ++queued;
  }
  void wait(long ticket) {
    std::unique_lock<std::mutex> lock(mu);
    cv.wait(lock, [&] { return done >= ticket; });
  }
};

struct Event {
  Stream* stream = nullptr;
  long ticket = 0;
};

inline Stream* of(hipStream_t s) { return reinterpret_cast<Stream*>(s); }
inline Event* of(hipEvent_t e) { return reinterpret_cast<Event*>(e); }
inline hipStream_t handle(Stream& s) { return reinterpret_cast<hipStream_t>(&s); }

inline void check(bool ok, const char* what) {
  if (ok) return;
  std::printf("FAILED: %s\n", what);
  std::exit(1);
}

}  // namespace fake

extern "C" {
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  if (fake::refuse_pinned) return hipErrorOutOfMemory;
  ++fake::pinned_allocations;
  ++fake::pinned_alive;
  *p = std::malloc(bytes);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  --fake::pinned_alive;
  std::free(p);
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "a fake error"; }
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(new fake::Event);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  delete fake::of(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  fake::of(e)->stream = fake::of(s);
  fake::of(e)->ticket = fake::of(s)->put([] {});
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  if (fake::of(e)->stream) fake::of(e)->stream->wait(fake::of(e)->ticket);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* to, const void* from, size_t bytes, hipMemcpyKind, hipStream_t s) {
  ++fake::copies;
  fake::of(s)->put([=] { std::memcpy(to, from, bytes); });
  return hipSuccess;
}
hipError_t hipMemcpy(void* to, const void* from, size_t bytes, hipMemcpyKind) {
  ++fake::copies;
  std::memcpy(to, from, bytes);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  fake::of(s)->wait(fake::of(s)->put([] {}));
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t s) {
  if (fake::stream_status >= 0) return static_cast<hipError_t>(fake::stream_status.load());
  std::lock_guard<std::mutex> lock(fake::of(s)->mu);
  return fake::of(s)->done == fake::of(s)->queued ? hipSuccess : hipErrorNotReady;
}
}
