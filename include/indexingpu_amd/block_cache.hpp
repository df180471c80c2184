// Device memory of closed indexes, kept for the next ones.
//
// The driver wipes every block that is freed, at about 41 GB/s (a 3.4 GB slab pool: 84 ms),
// first in the background and, once the backlog fills the card, in the way of the next
// allocation: a program that makes, loads and closes indexes in turn ran at the wipe's rate
// (16M-key loads of 19 ms of GPU work took 45 to 130 ms).  Blocks of 1 MB or more therefore
// go to a list and serve the next allocation of about their size.
//
// Bounded: at most 1/32 of the device's memory is kept per process and device (9 GB of 288);
// larger blocks, and the oldest ones beyond that, are freed at once.  Given back: a block not
// taken again within kMaxAge allocations is freed, every block is when an allocation of this
// library fails, and release_kept() (gmt_release_memory) frees all of them.  Thread-safe; the
// device is idle with respect to a block before it is kept, as hipFree waits for it too.
#pragma once
#include <cstdint>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "hip_util.hpp"

namespace indexingpu_amd {

class block_cache {
 public:
  static block_cache& instance() {
    static block_cache* c = new block_cache;  // never destroyed: indexes may outlive statics
    return *c;
  }

  hipError_t take(void** out, std::size_t bytes) {
    *out = nullptr;
    if (bytes < kMinBytes) return hipMalloc(out, bytes);
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> g(mu_);
    clock_ += 1;
    std::size_t best = kept_.size();
    for (std::size_t i = 0; i < kept_.size(); i++) {
      const block& b = kept_[i];
      if (b.dev == dev && b.bytes >= bytes && b.bytes - bytes <= bytes / 4 &&
          (best == kept_.size() || b.bytes < kept_[best].bytes))
        best = i;
    }
    if (best < kept_.size()) {
      *out = kept_[best].ptr;
      live_[*out] = {dev, kept_[best].bytes};
      drop(best, false);
      return hipSuccess;
    }
    for (std::size_t i = kept_.size(); i-- > 0;)
      if (clock_ - kept_[i].since > kMaxAge) drop(i, true);
    e = hipMalloc(out, bytes);
    if (e != hipSuccess && !kept_.empty()) {
      (void)hipGetLastError();
      release_locked();
      e = hipMalloc(out, bytes);
    }
    if (e == hipSuccess) live_[*out] = {dev, bytes};
    return e;
  }

  void give(void* ptr) {
    if (!ptr) return;
    std::unique_lock<std::mutex> g(mu_);
    auto it = live_.find(ptr);
    if (it == live_.end()) {  // a small block
      g.unlock();
      (void)hipFree(ptr);
      return;
    }
    const live_block l = it->second;
    live_.erase(it);
    g.unlock();
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (dev != l.dev) (void)hipSetDevice(l.dev);
    const bool idle = hipDeviceSynchronize() == hipSuccess;
    std::size_t free_b = 0, total_b = 0;
    const bool known = hipMemGetInfo(&free_b, &total_b) == hipSuccess;
    if (dev != l.dev) (void)hipSetDevice(dev);
    const std::size_t most = total_b / 32;
    g.lock();
    if (!idle || !known || l.bytes > most) {
      (void)hipFree(ptr);
      return;
    }
    while (!kept_.empty() && kept_bytes(l.dev) + l.bytes > most) drop(oldest(l.dev), true);
    kept_.push_back({ptr, l.dev, l.bytes, clock_});
  }

  void release() {
    std::lock_guard<std::mutex> g(mu_);
    release_locked();
  }

 private:
  static constexpr std::size_t kMinBytes = 1u << 20;
  static constexpr uint64_t kMaxAge = 64;
  struct block {
    void* ptr;
    int dev;
    std::size_t bytes;
    uint64_t since;
  };
  struct live_block {
    int dev;
    std::size_t bytes;
  };
  std::size_t kept_bytes(int dev) const {
    std::size_t s = 0;
    for (const block& b : kept_) s += b.dev == dev ? b.bytes : 0;
    return s;
  }
  std::size_t oldest(int dev) const {  // kept_ is in order of age
    for (std::size_t i = 0; i < kept_.size(); i++)
      if (kept_[i].dev == dev) return i;
    return 0;
  }
  void drop(std::size_t i, bool free_it) {
    if (free_it) (void)hipFree(kept_[i].ptr);
    kept_.erase(kept_.begin() + (std::ptrdiff_t)i);
  }
  void release_locked() {
    while (!kept_.empty()) drop(kept_.size() - 1, true);
  }
  std::mutex mu_;
  std::vector<block> kept_;
  std::unordered_map<void*, live_block> live_;
  uint64_t clock_ = 0;
};

template <class T>
inline hipError_t device_take(T** out, std::size_t bytes) {
  return block_cache::instance().take(reinterpret_cast<void**>(out), bytes);
}
inline void device_give(void* ptr) { block_cache::instance().give(ptr); }
inline void release_kept() { block_cache::instance().release(); }

}  // namespace indexingpu_amd
