// transfer.hip -- see transfer.h.
#include "transfer.h"

#include <atomic>
#include <cstring>
#include <thread>

namespace cube {

namespace {
// An ordinary pointer: none the runtime knows (pinned, managed or device memory goes its way).
bool pageable(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return true;
}
}  // namespace

Transfers::~Transfers() {
  for (Lane& l : lane_)
    for (int k = 0; k < 2; ++k) {
      if (l.ev[k]) {
        (void)hipEventSynchronize(l.ev[k]);
        (void)hipEventDestroy(l.ev[k]);
      }
      if (l.buf[k]) (void)hipHostFree(l.buf[k]);
    }
}

// The lanes' buffers and events; false if there is no memory for them.
bool Transfers::make() {
  for (Lane& l : lane_)
    for (int k = 0; k < 2; ++k) {
      if (!l.ev[k] && hipEventCreateWithFlags(&l.ev[k], hipEventDisableTiming) != hipSuccess) l.ev[k] = nullptr;
      if (!l.buf[k] && hipHostMalloc((void**)&l.buf[k], kChunk, hipHostMallocDefault) != hipSuccess) l.buf[k] = nullptr;
      if (!l.ev[k] || !l.buf[k]) {
        (void)hipGetLastError();
        return false;
      }
    }
  return true;
}

// fn(lane) on kLanes threads, the caller's among them; the first error is thrown
// when all have ended.
template <class Fn>
void Transfers::run(Fn&& fn) {
  int device = 0;
  CUBE_HIP(hipGetDevice(&device));
  std::atomic<int> rc{(int)hipSuccess};
  auto body = [&](int i) {
    hipError_t e = hipSetDevice(device);
    if (e == hipSuccess) e = fn(lane_[i], (size_t)i);
    int none = (int)hipSuccess;
    if (e != hipSuccess) rc.compare_exchange_strong(none, (int)e);
  };
  std::thread th[kLanes];
  for (int i = 1; i < kLanes; ++i) {
    try {
      th[i] = std::thread(body, i);
    } catch (const std::exception&) {  // no thread to be had: the lane's share runs below
    }
  }
  body(0);
  for (int i = 1; i < kLanes; ++i) {
    if (th[i].joinable()) th[i].join();
    else body(i);
  }
  CUBE_HIP((hipError_t)rc.load());
}

void Transfers::in(void* dev, const void* host, size_t bytes, hipStream_t s) {
  if (bytes < kStageFrom || !pageable(host) || !make()) {
    CUBE_HIP(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s));
    return;
  }
  const size_t step = chunk(bytes), n = (bytes + step - 1) / step;
  run([&](Lane& l, size_t i) {
    int k = 0;
    for (size_t c = i; c < n; c += kLanes, k ^= 1) {
      const size_t at = c * step, len = std::min(step, bytes - at);
      hipError_t e = hipEventSynchronize(l.ev[k]);  // the buffer's last copy (of an earlier call, too)
      if (e != hipSuccess) return e;
      std::memcpy(l.buf[k], (const char*)host + at, len);
      e = hipMemcpyAsync((char*)dev + at, l.buf[k], len, hipMemcpyHostToDevice, s);
      if (e == hipSuccess) e = hipEventRecord(l.ev[k], s);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  });
}

void Transfers::out(void* host, const void* dev, size_t bytes, hipStream_t s) {
  if (bytes < kStageFrom || !pageable(host) || !make()) {
    CUBE_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s));
    return;
  }
  const size_t step = chunk(bytes), n = (bytes + step - 1) / step;
  run([&](Lane& l, size_t i) {
    auto queue = [&](size_t c, int k) {
      const size_t at = c * step, len = std::min(step, bytes - at);
      hipError_t e = hipEventSynchronize(l.ev[k]);  // the buffer's last copy
      if (e == hipSuccess) e = hipMemcpyAsync(l.buf[k], (const char*)dev + at, len, hipMemcpyDeviceToHost, s);
      if (e == hipSuccess) e = hipEventRecord(l.ev[k], s);
      return e;
    };
    hipError_t e = hipSuccess;
    for (int k = 0; k < 2 && e == hipSuccess; ++k)
      if (i + k * kLanes < n) e = queue(i + k * kLanes, k);
    int k = 0;
    for (size_t c = i; c < n && e == hipSuccess; c += kLanes, k ^= 1) {
      e = hipEventSynchronize(l.ev[k]);
      if (e != hipSuccess) break;
      std::memcpy((char*)host + c * step, l.buf[k], std::min(step, bytes - c * step));
      if (c + 2 * kLanes < n) e = queue(c + 2 * kLanes, k);
    }
    return e;
  });
}

char* PinnedPage::get() {
  if (!p) CUBE_HIP(hipHostMalloc((void**)&p, kBytes, hipHostMallocDefault));
  return p;
}
PinnedPage::~PinnedPage() {
  if (p) (void)hipHostFree(p);
}

// Copies that nobody waited for (an error on the way) end before the page is used again.
ReadBack::~ReadBack() {
  if (pending_) (void)hipStreamSynchronize(s_);
}

void ReadBack::get(void* dst, const void* dev, size_t bytes, hipStream_t s) {
  s_ = s;
  pending_ = true;
  if (used_ + bytes > PinnedPage::kBytes) {
    CUBE_HIP(hipMemcpyAsync(dst, dev, bytes, hipMemcpyDeviceToHost, s));
    return;
  }
  CUBE_HIP(hipMemcpyAsync(page_.get() + used_, dev, bytes, hipMemcpyDeviceToHost, s));
  items_.push_back({dst, used_, bytes});
  used_ += (bytes + 63) / 64 * 64;
}

void ReadBack::wait() {
  CUBE_HIP(hipStreamSynchronize(s_));
  pending_ = false;
  for (const Item& i : items_) std::memcpy(i.dst, page_.p + i.at, i.bytes);
  items_.clear();
  used_ = 0;
}

}  // namespace cube
