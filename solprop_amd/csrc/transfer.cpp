// Pipelined copies of large pageable fields (see transfer.hpp).
#include "transfer.hpp"

#include <algorithm>
#include <cstring>
#include <exception>
#include <system_error>
#include <thread>

namespace sp {

Transfer::~Transfer() {
  for (auto& e : events_)
    if (e) (void)hipEventDestroy(e);
  if (slots_) (void)hipHostFree(slots_);
}

void Transfer::make_slots() {
  void* p = nullptr;
  bool ok = hipHostMalloc(&p, kLanes * kSlots * kChunk) == hipSuccess;
  for (auto& e : events_)
    ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
  if (ok) {
    slots_ = static_cast<char*>(p);
    return;
  }
  if (p) (void)hipHostFree(p);
  (void)hipGetLastError();
  failed_ = true;
}

// Whether a download of `bytes` goes through the slots, which it makes when they pay.
bool Transfer::slots_for(std::size_t bytes) {
  if (slots_ || failed_ || bytes < kDownload) return slots_ && bytes >= kDownload;
  if (bytes >= kAtOnce || plain_ >= kRepaid) make_slots();
  if (!slots_) plain_ += bytes;
  return slots_ != nullptr;
}

// Runs lane(0) .. lane(kLanes - 1), each on a thread of its own where one can be had, and
// throws the first lane's exception after all have ended.
template <typename F>
void Transfer::run(F&& lane) {
  int device = 0;
  SP_HIP(hipGetDevice(&device));
  std::exception_ptr errors[kLanes];
  auto guarded = [&](int i) noexcept {
    try {
      SP_HIP(hipSetDevice(device));
      lane(i);
    } catch (...) {
      errors[i] = std::current_exception();
    }
  };
  std::thread threads[kLanes];
  for (int i = 1; i < kLanes; ++i) {
    try {
      threads[i] = std::thread(guarded, i);
    } catch (const std::system_error&) {
      guarded(i);
    }
  }
  guarded(0);
  for (auto& t : threads)
    if (t.joinable()) t.join();
  for (auto& e : errors)
    if (e) std::rethrow_exception(e);
}

void Transfer::upload(void* device, const void* host, std::size_t bytes, hipStream_t stream) {
  if (bytes < kUpload || !slots_) {
    SP_HIP(hipStreamSynchronize(stream));
    SP_HIP(hipMemcpy(device, host, bytes, hipMemcpyHostToDevice));
    return;
  }
  const std::size_t chunks = (bytes + kChunk - 1) / kChunk;
  run([&](int lane) {
    int n = 0;
    for (std::size_t c = lane; c < chunks; c += kLanes, ++n) {
      const int at = lane * kSlots + n % kSlots;
      char* slot = slots_ + at * kChunk;
      const std::size_t size = std::min(kChunk, bytes - c * kChunk);
      if (n >= kSlots) SP_HIP(hipEventSynchronize(events_[at]));
      std::memcpy(slot, static_cast<const char*>(host) + c * kChunk, size);
      SP_HIP(hipMemcpyAsync(static_cast<char*>(device) + c * kChunk, slot, size,
                            hipMemcpyHostToDevice, stream));
      SP_HIP(hipEventRecord(events_[at], stream));
    }
  });
  SP_HIP(hipStreamSynchronize(stream));
}

void Transfer::download(void* host, const void* device, std::size_t bytes, hipStream_t stream) {
  if (!slots_for(bytes)) {
    SP_HIP(hipStreamSynchronize(stream));
    SP_HIP(hipMemcpy(host, device, bytes, hipMemcpyDeviceToHost));
    return;
  }
  const std::size_t chunks = (bytes + kChunk - 1) / kChunk;
  run([&](int lane) {
    auto slot_at = [&](int n) { return lane * kSlots + n % kSlots; };
    auto fetch = [&](std::size_t c, int n) {
      const std::size_t size = std::min(kChunk, bytes - c * kChunk);
      SP_HIP(hipMemcpyAsync(slots_ + slot_at(n) * kChunk,
                            static_cast<const char*>(device) + c * kChunk, size,
                            hipMemcpyDeviceToHost, stream));
      SP_HIP(hipEventRecord(events_[slot_at(n)], stream));
    };
    int n = 0;
    if (static_cast<std::size_t>(lane) < chunks) fetch(lane, 0);
    for (std::size_t c = lane; c < chunks; c += kLanes, ++n) {
      if (c + kLanes < chunks) fetch(c + kLanes, n + 1);
      SP_HIP(hipEventSynchronize(events_[slot_at(n)]));
      std::memcpy(static_cast<char*>(host) + c * kChunk, slots_ + slot_at(n) * kChunk,
                  std::min(kChunk, bytes - c * kChunk));
    }
  });
  SP_HIP(hipStreamSynchronize(stream));
}

}  // namespace sp
