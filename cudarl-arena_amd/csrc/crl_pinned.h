// Pinned host memory that kernels read and write in place.
//
// A small call is all latency: one launch whose kernel stores its results and a
// sequence number straight into host memory answers in 6.3 us (MI355X, launch to
// the host's seeing the number), the same launch followed by hipStreamSynchronize
// in 10.9 us, and every copy to or from pageable memory adds 10 to 20 us of its
// own.  A kernel moves 55 GB/s over the link in either direction, as much as a
// copy engine, so nothing is lost on large calls either.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>
#include <utility>
#include <vector>

namespace crl {

// Blocks of pinned, device-mapped, coherent host memory, rounded up to a power of two.
// Pinning costs far more than a call that uses the block (the driver maps it into the
// GPU's page tables), so blocks of destroyed engines are kept for later ones: at most
// kHeldBytes of them, and none once the last engine of the process is gone.
class PinnedPool {
 public:
  static PinnedPool& get() {
    static PinnedPool* pool = new PinnedPool();  // (never destroyed: the HIP runtime may be gone before it)
    return *pool;
  }
  void add_user() {
    std::lock_guard<std::mutex> hold(lock_);
    ++users_;
  }
  void drop_user() {
    std::lock_guard<std::mutex> hold(lock_);
    if (--users_ == 0) {
      for (auto& b : free_) (void)hipHostFree(b.second);
      free_.clear();
      held_ = 0;
    }
  }
  // -> a block of at least `bytes`, its size in *got; null if there is none
  void* take(size_t bytes, size_t* got) {
    size_t size = kMinBytes;
    while (size < bytes) size *= 2;
    {
      std::lock_guard<std::mutex> hold(lock_);
      for (size_t i = 0; i < free_.size(); ++i)
        if (free_[i].first == size) {
          void* p = free_[i].second;
          free_[i] = free_.back();
          free_.pop_back();
          held_ -= size;
          *got = size;
          return p;
        }
    }
    void* p = nullptr;
    if (hipHostMalloc(&p, size, hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    *got = size;
    return p;
  }
  void give(void* p, size_t size) {
    {
      std::lock_guard<std::mutex> hold(lock_);
      if (users_ > 0 && held_ + size <= kHeldBytes) {
        try {
          free_.emplace_back(size, p);
          held_ += size;
          return;
        } catch (...) {  // no room in the list: give the block back below
        }
      }
    }
    (void)hipHostFree(p);
  }

 private:
  static constexpr size_t kMinBytes = 4096;
  static constexpr size_t kHeldBytes = (size_t)64 << 20;
  std::mutex lock_;
  std::vector<std::pair<size_t, void*>> free_;
  size_t held_ = 0;
  int users_ = 0;
};

// A block of the pool that belongs to one engine.  Grows, never shrinks; growing drops
// the contents, so only while no kernel works on it.
struct PinBuf {
  unsigned char* p = nullptr;
  size_t n = 0;
  bool ensure(size_t bytes) {
    if (bytes <= n) return true;
    release();
    p = static_cast<unsigned char*>(PinnedPool::get().take(bytes, &n));
    if (!p) n = 0;
    return p != nullptr;
  }
  void release() {
    if (p) PinnedPool::get().give(p, n);
    p = nullptr;
    n = 0;
  }
  ~PinBuf() { release(); }
  PinBuf() = default;
  PinBuf(const PinBuf&) = delete;
  PinBuf& operator=(const PinBuf&) = delete;
};

}  // namespace crl
