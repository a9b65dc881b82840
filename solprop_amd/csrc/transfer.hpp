// Large fields between a caller's pageable memory and the device.
//
// A plain copy into pageable memory is one host thread's: it moves 17 GB/s, 10 where the
// destination's pages are touched for the first time (every array above the C library's
// 32 MB threshold). Here kLanes host threads copy chunks through pinned slots of their
// own, two each, so that the page faults, the host copies and the link overlap. State of
// 8.4, 16.8, 33.6, 67 and 268 MB to the host, plain and in lanes: 0.49 and 0.36 ms, 1.02
// and 0.62, 3.35 and 1.30, 6.8 and 2.4, 25.6 and 9.1. From pageable memory the plain copy
// is as quick as the link but for the largest: 0.24 and 0.33, 0.46 and 0.60, 1.15 and 1.14,
// 2.26 and 2.20, 8.95 and 8.52 ms.
//
// The slots take 1.1 to 1.5 ms to make (a process's first pinned copy 5 ms more), so they
// are made when they pay: by a field of 32 MB (its own copy repays them), or when fields of
// 8 MB and more have come back by plain copies to 64 MB in all, which have then lost as
// much. Below 32 MB a workspace that is loaded and read once copies as if there were none.
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

  // Both order the copy after what `stream` holds and return when it is done. Where the
  // slots do not pay or cannot be had, the copy is a plain one.
  void upload(void* device, const void* host, std::size_t bytes, hipStream_t stream);
  void download(void* host, const void* device, std::size_t bytes, hipStream_t stream);

 private:
  static constexpr int kLanes = 4;
  static constexpr int kSlots = 2;                   // a lane
  static constexpr std::size_t kChunk = 1UL << 20;   // bytes of a slot
  static constexpr std::size_t kDownload = 8UL << 20;  // the least that lanes are quicker for
  static constexpr std::size_t kUpload = 32UL << 20;   // and the least to the device
  static constexpr std::size_t kAtOnce = 32UL << 20;   // a download that repays the slots
  static constexpr std::size_t kRepaid = 64UL << 20;   // plain downloads that would have
  bool slots_for(std::size_t bytes);
  void make_slots();
  template <typename F>
  void run(F&& lane);
  char* slots_ = nullptr;  // (kLanes, kSlots, kChunk) pinned
  hipEvent_t events_[kLanes * kSlots] = {};
  std::size_t plain_ = 0;  // bytes downloaded without slots, of fields they would speed up
  bool failed_ = false;
};

}  // namespace sp
