// Device buffers handed to callers (cuhc_device_alloc, cuhc_device_free).
//
// A fresh 335 MB buffer costs 0.4 ms of page mapping, more than the distance
// matrix that fills it, so freed buffers are kept for the next request of the
// same size on the same device, apart from the library's own cache of blocks.
// Device is the runtime under it (the HIP runtime; a stand-in in the tests).
// What it promises callers:
//   - a freed buffer is kept only after its own device has finished everything
//     that was queued when it was freed, on every stream, as hipFree waits;
//   - freeing a buffer a second time is an error, as for hipFree, and frees
//     nothing; a pointer that is no buffer of this pool goes to the runtime;
//   - at most Device::keepLimit() bytes are kept, the oldest making way, and
//     given back by releaseKept(), which also runs where an allocation finds no
//     memory.
// No HIP types here: the file compiles on the host alone.
#pragma once

#include "kept_blocks.hpp"

#include <stddef.h>

#include <mutex>
#include <new>
#include <unordered_map>
#include <utility>

namespace cuhc {

// The HIP statuses that the pool itself returns or acts on.
constexpr int kStatusInvalidValue = 1;
constexpr int kStatusOutOfMemory = 2;

template <class Device> class CallerBuffers {
public:
  explicit CallerBuffers(Device device = Device{}) : device_(device) {}

  int alloc(void **ptr, size_t bytes) {
    *ptr = nullptr;
    int on = 0;
    if (const int s = device_.current(&on))
      return s;
    void *p = takeKept(on, bytes);
    if (p) {
      *ptr = p;
      return 0;
    }
    int s = device_.allocate(&p, bytes);
    if (s == kStatusOutOfMemory) {
      releaseKept();
      device_.releaseOther();
      s = device_.allocate(&p, bytes);
    }
    if (s || !p) // no bytes: no buffer
      return s;
    try {
      std::lock_guard<std::mutex> lock(mutex_);
      buffers_[p] = Buffer{on, bytes, true};
    } catch (const std::bad_alloc &) {
      (void)device_.release(p);
      return kStatusOutOfMemory;
    }
    *ptr = p;
    return 0;
  }

  int free(void *ptr) {
    if (!ptr)
      return 0;
    Buffer b;
    bool known = false;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      const auto it = buffers_.find(ptr);
      if (it != buffers_.end()) {
        if (!it->second.held)
          return kStatusInvalidValue; // freed before
        it->second.held = false;
        b = it->second;
        known = true;
      }
    }
    if (!known)
      return device_.release(ptr);
    const int s = device_.wait(b.device);
    // A buffer that the runtime no longer holds (freed past this pool) is an error below.
    if (s == 0 && device_.covers(ptr, b.bytes) && keep(ptr, b))
      return 0;
    // Perhaps still in use, or no room: not for the next call.
    {
      std::lock_guard<std::mutex> lock(mutex_);
      buffers_.erase(ptr);
    }
    const int freed = device_.release(ptr);
    return s ? s : freed;
  }

  void releaseKept() {
    std::lock_guard<std::mutex> lock(mutex_);
    kept_.clear([this](void *p) { forget(p); });
  }

  size_t keptBytes() {
    std::lock_guard<std::mutex> lock(mutex_);
    return kept_.bytes();
  }

private:
  struct Buffer {
    int device = 0;
    size_t bytes = 0;
    bool held = false; // by a caller; otherwise kept, or on its way there
  };
  using Key = std::pair<int, size_t>; // device, bytes

  void *takeKept(int on, size_t bytes) {
    std::lock_guard<std::mutex> lock(mutex_);
    void *p = kept_.take(Key{on, bytes});
    if (p)
      buffers_[p].held = true;
    return p;
  }

  bool keep(void *p, const Buffer &b) {
    const size_t limit = device_.keepLimit();
    std::lock_guard<std::mutex> lock(mutex_);
    return kept_.put(Key{b.device, b.bytes}, p, b.bytes, limit, [this](void *q) { forget(q); });
  }

  void forget(void *p) {
    buffers_.erase(p);
    (void)device_.release(p);
  }

  Device device_;
  std::mutex mutex_;
  std::unordered_map<void *, Buffer> buffers_; // handed out, or kept
  KeptBlocks<Key> kept_;
};

} // namespace cuhc
