// Device memory kept between its owners.
#ifndef DFTGRID_DEVICE_POOL_H
#define DFTGRID_DEVICE_POOL_H

#include <cstddef>
#include <map>
#include <mutex>
#include <unordered_map>
#include <utility>

namespace dg {

// Blocks that were given, for the next taker of about the same size on the same
// device; at most `most` bytes, those kept longest leaving first.  Api has the static
// members device(int*), alloc(void**, size_t) (0: done), release(void*) and the error
// code kNoMemory.  Nothing is thrown: a block that cannot be recorded goes back.
// A kept block is found in the time of a map's look-up (through a list of all blocks,
// a program that closes many small handles paid for each of them on every allocation).
template <typename Api>
class DevicePool {
 public:
  explicit DevicePool(size_t most) : most_(most) {}

  int take(void** p, size_t bytes) noexcept {
    *p = nullptr;
    bytes = bytes < 512 ? 512 : (bytes + 511) / 512 * 512;
    int dev = 0;
    if (const int e = Api::device(&dev)) return e;
    {
      std::lock_guard<std::mutex> lock(m_);
      const auto it = kept_.lower_bound(Size{dev, bytes});
      if (it != kept_.end() && it->first.first == dev && it->first.second <= bytes + bytes / 8) {
        if (!use(it->second.p, it->first)) return Api::kNoMemory;
        *p = it->second.p;
        forget(it);
        return 0;
      }
    }
    if (const int e = raw(p, bytes)) return e;
    std::lock_guard<std::mutex> lock(m_);
    if (use(*p, Size{dev, bytes})) return 0;
    Api::release(*p);
    *p = nullptr;
    return Api::kNoMemory;
  }

  // For work that is over on every stream.
  void give(void* p) noexcept {
    if (!p) return;
    std::lock_guard<std::mutex> lock(m_);
    const auto it = used_.find(p);
    if (it == used_.end()) return;
    const Size s = it->second;
    used_.erase(it);
    while (s.second <= most_ && held_ + s.second > most_) drop_oldest();
    if (s.second > most_ || !keep(p, s)) Api::release(p);
  }

  // A block of the caller's own, not to be given: straight from the device, the kept
  // blocks going back to it first if it has no room.
  int raw(void** p, size_t bytes) noexcept {
    int e = Api::alloc(p, bytes);
    if (e && release_kept()) e = Api::alloc(p, bytes);
    if (e) *p = nullptr;
    return e;
  }

  // All kept blocks go back to the device; whether there were any.
  bool release_kept() noexcept {
    std::lock_guard<std::mutex> lock(m_);
    const bool any = !kept_.empty();
    while (!kept_.empty()) drop_oldest();
    return any;
  }

 private:
  using Size = std::pair<int, size_t>;  // device, bytes
  struct Kept {
    void* p;
    unsigned long age;
  };
  using Blocks = std::multimap<Size, Kept>;

  bool use(void* p, Size s) noexcept {
    try {
      used_.emplace(p, s);
      return true;
    } catch (...) {
      return false;
    }
  }
  bool keep(void* p, Size s) noexcept {
    typename Blocks::iterator it = kept_.end();
    try {
      it = kept_.emplace(s, Kept{p, age_});
      by_age_.emplace(age_, it);
    } catch (...) {
      if (it != kept_.end()) kept_.erase(it);
      return false;
    }
    ++age_;
    held_ += s.second;
    return true;
  }
  void forget(typename Blocks::iterator it) noexcept {
    held_ -= it->first.second;
    by_age_.erase(it->second.age);
    kept_.erase(it);
  }
  void drop_oldest() noexcept {
    const auto it = by_age_.begin()->second;
    Api::release(it->second.p);
    forget(it);
  }

  const size_t most_;
  std::mutex m_;
  Blocks kept_;
  std::map<unsigned long, typename Blocks::iterator> by_age_;  // oldest first
  std::unordered_map<void*, Size> used_;
  size_t held_ = 0;
  unsigned long age_ = 0;
};

}  // namespace dg

#endif
