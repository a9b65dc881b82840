// Large fields between a caller's pageable memory and the device.
//
// A plain hipMemcpy of pageable memory moves 16 GB/s (one host thread copies through the
// runtime's staging, and a fresh destination's pages are first touched by it): on the
// free-space beam, 268 MB a field, the two copies took 34 ms beside 60 ms of kernels. Here
// kLanes host threads copy chunks through pinned slots of their own, two each, so that the
// host copies, the page faults and the link overlap: 31 GB/s, 17.5 ms. From 8 MB on the
// threads' start (0.1 ms) is well repaid.
#pragma once

#include <cstddef>

#include "common.hpp"

namespace sp {

class Transfer {
 public:
  Transfer() = default;
  ~Transfer();
  Transfer(const Transfer&) = delete;
  Transfer& operator=(const Transfer&) = delete;

  // Both order the copy after what `stream` holds and return when it is done. Fields
  // below kLeast bytes, and any where the slots cannot be had, take one plain copy.
  void upload(void* device, const void* host, std::size_t bytes, hipStream_t stream);
  void download(void* host, const void* device, std::size_t bytes, hipStream_t stream);

 private:
  static constexpr int kLanes = 4;
  static constexpr int kSlots = 2;                     // a lane
  static constexpr std::size_t kChunk = 1UL << 20;     // bytes of a slot
  static constexpr std::size_t kLeast = 8UL << 20;
  bool ready();
  template <typename F>
  void run(F&& lane);
  char* slots_ = nullptr;  // (kLanes, kSlots, kChunk) pinned, from the first large copy on
  hipEvent_t events_[kLanes * kSlots] = {};
  bool failed_ = false;
};

}  // namespace sp
