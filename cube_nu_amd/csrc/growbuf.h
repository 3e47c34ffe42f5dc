// growbuf.h -- arrays that grow with the calls, and outlive their growth where a
// captured call has used them.
#pragma once
#include <cstddef>
#include <vector>

namespace cube {

// An array of the memory that Mem gives (alloc throws when there is none).  A HIP
// graph holds the addresses that its calls used, so an array a captured call has
// used (hold) is not freed when a later call needs a larger one: it is kept beside
// the new one until the owner ends, and the graph may be replayed until then.
template <typename T, class Mem>
struct GrowBuf {
  T* p = nullptr;
  std::size_t n = 0;
  GrowBuf() = default;
  GrowBuf(const GrowBuf&) = delete;
  GrowBuf& operator=(const GrowBuf&) = delete;
  ~GrowBuf() {
    if (p) Mem::free(p);
    for (T* q : kept_) Mem::free(q);
  }
  T* ensure(std::size_t m) {
    if (m > n) {
      if (held_) kept_.push_back(p);
      else if (p) Mem::free(p);
      held_ = false;
      p = nullptr;
      n = 0;
      p = static_cast<T*>(Mem::alloc(m * sizeof(T)));
      n = m;
    }
    return p;
  }
  void hold() { held_ = p != nullptr; }

 private:
  bool held_ = false;
  std::vector<T*> kept_;
};

}  // namespace cube
