// Host-side synchronisation helpers: graph capture that always ends, and a bounded wait.
#pragma once

#include <algorithm>
#include <chrono>
#include <cstdint>
#include <string>
#include <thread>

#include "common.hpp"

namespace sp {

// Capture what `enqueue` puts on `stream` into an executable graph. If `enqueue` throws
// (a refused shape, a launch error), the capture is ended and its partial graph
// destroyed before the exception goes on, so the stream leaves capture mode and later
// calls on it work.
template <typename F>
hipGraphExec_t capture_graph(hipStream_t stream, F&& enqueue) {
  SP_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
  try {
    enqueue();
  } catch (...) {
    hipGraph_t partial = nullptr;
    if (hipStreamEndCapture(stream, &partial) == hipSuccess && partial)
      (void)hipGraphDestroy(partial);
    (void)hipGetLastError();
    throw;
  }
  hipGraph_t graph = nullptr;
  SP_HIP(hipStreamEndCapture(stream, &graph));
  hipGraphExec_t exec = nullptr;
  const hipError_t made = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  SP_HIP(made);
  return exec;
}

// How long a wait for the device may take before it is reported as a failure, seconds.
constexpr double kWaitLimitSeconds = 300.0;

// Wait until `event` completes: spin for the first `spin_us` microseconds (a trial's
// norms are wanted as soon as they land), then yield the core, then sleep for a 32nd of
// the time waited so far, up to a millisecond: the event is seen at most 3 % late, and by
// what the host's timers add to a sleep (some 50 us). (Steps that doubled from 2 us
// overslept a 2.4 ms step by 0.9 ms.) A wait past kWaitLimitSeconds throws SP_BACKEND, so a
// device that never finishes cannot hold the host forever.
inline void wait_event(hipEvent_t event, double spin_us = 200.0) {
  using clock = std::chrono::steady_clock;
  const auto start = clock::now();
  for (;;) {
    const hipError_t status = hipEventQuery(event);
    if (status == hipSuccess) return;
    if (status != hipErrorNotReady) SP_HIP(status);
    const double waited =
        std::chrono::duration<double, std::micro>(clock::now() - start).count();
    if (waited < spin_us) continue;
    if (waited > kWaitLimitSeconds * 1e6)
      throw Error(kBackend, "the device did not finish within " +
                                std::to_string(static_cast<int>(kWaitLimitSeconds)) + " s");
    if (waited < 4.0 * spin_us) {
      std::this_thread::yield();
      continue;
    }
    std::this_thread::sleep_for(
        std::chrono::duration<double, std::micro>(std::min(waited / 32.0, 1000.0)));
  }
}

// A trial's sums in mapped host memory, awaited by their values: a kernel stores each of
// them once, at system scope (store_awaited), and the host sees them when they land, some
// 5 us before an event after the kernel reports its end. `expect_sums` fills them with a
// NaN that no arithmetic makes before the launch; `wait_sums` returns once none is left,
// and while it waits beyond `spin_us` asks the stream for errors, as wait_event does. The
// kernel may still be ending then: later work on the stream follows it.
constexpr std::uint64_t kAwaited = 0x7ff4a3c15e97d2b6ULL;  // a signalling NaN

inline void expect_sums(double* sums, int n) {
  for (int i = 0; i < n; ++i)
    __atomic_store_n(reinterpret_cast<std::uint64_t*>(sums) + i, kAwaited, __ATOMIC_RELAXED);
  __atomic_thread_fence(__ATOMIC_SEQ_CST);
}

inline void wait_sums(const double* sums, int n, hipStream_t stream, double spin_us = 200.0) {
  using clock = std::chrono::steady_clock;
  const auto start = clock::now();
  int at = 0;
  auto landed = [&] {
    while (at < n && __atomic_load_n(reinterpret_cast<const std::uint64_t*>(sums) + at,
                                     __ATOMIC_ACQUIRE) != kAwaited)
      ++at;
    return at == n;
  };
  for (;;) {
    if (landed()) return;
    const double waited =
        std::chrono::duration<double, std::micro>(clock::now() - start).count();
    if (waited < spin_us) continue;
    const hipError_t status = hipStreamQuery(stream);
    if (status == hipSuccess) {
      if (landed()) return;
      throw Error(kBackend, "the device ended a trial without its sums");
    }
    if (status != hipErrorNotReady) SP_HIP(status);
    if (waited > kWaitLimitSeconds * 1e6)
      throw Error(kBackend, "the device did not finish within " +
                                std::to_string(static_cast<int>(kWaitLimitSeconds)) + " s");
    if (waited < 4.0 * spin_us) {
      std::this_thread::yield();
      continue;
    }
    std::this_thread::sleep_for(
        std::chrono::duration<double, std::micro>(std::min(waited / 32.0, 1000.0)));
  }
}

}  // namespace sp
