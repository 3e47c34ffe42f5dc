// transfer.h -- copies between host programs' arrays and the device.
//
// Host programs hand over ordinary (pageable) arrays, which the copy engine
// cannot read: their bytes pass through pinned memory.  The runtime's own staging
// is one thread's copy; here kLanes threads each copy every kLanes-th chunk through
// two pinned buffers of their own while the engine moves the other.  Pinned arrays,
// and those below kStageFrom, take the runtime's path.  302 MB in 6.4 ms and 201 MB
// out 4.4 (PCIe 5.3 and 3.5; 2 MB chunks on eight lanes 7.7 and 5.2, the runtime's
// staging 17 in all more).
#pragma once
#include "common.h"

namespace cube {

class Transfers {
 public:
  ~Transfers();
  // host -> device, queued on s.  An array that is staged may change when it returns;
  // one the runtime copies itself (pinned, managed, small) only once s has come that
  // far: the caller synchronises before it gives such an array back
  void in(void* dev, const void* host, size_t bytes, hipStream_t s);
  // device -> host after what s holds; the array is complete once s is synchronised
  void out(void* host, const void* dev, size_t bytes, hipStream_t s);

 private:
  static constexpr int kLanes = 4;
  static constexpr size_t kChunk = (size_t)8 << 20;  // 64 MB of pinned memory a context, from its first use on
  static constexpr size_t kStageFrom = (size_t)8 << 20;
  // two chunks a lane where the array is small
  static size_t chunk(size_t bytes) {
    const size_t c = (bytes / (2 * kLanes) + ((size_t)1 << 20)) >> 20 << 20;
    return c < kChunk ? c : kChunk;
  }
  struct Lane {
    char* buf[2] = {nullptr, nullptr};
    hipEvent_t ev[2] = {nullptr, nullptr};
  } lane_[kLanes];
  bool make();
  template <class Fn>
  void run(Fn&& fn);
};

// A page of pinned memory for small results.
struct PinnedPage {
  static constexpr size_t kBytes = (size_t)64 << 10;
  char* p = nullptr;
  char* get();
  ~PinnedPage();
};

// Small results read back together: get() queues the copies into a pinned page,
// wait() synchronises once and hands them out (a copy to pageable memory stops the
// host each time: 20 us).  One at a time for a page.
class ReadBack {
 public:
  explicit ReadBack(PinnedPage& page) : page_(page) {}
  ~ReadBack();
  void get(void* dst, const void* dev, size_t bytes, hipStream_t s);
  void wait();

 private:
  struct Item {
    void* dst;
    size_t at, bytes;
  };
  PinnedPage& page_;
  size_t used_ = 0;
  std::vector<Item> items_;
  hipStream_t s_ = nullptr;
  bool pending_ = false;
};

}  // namespace cube
