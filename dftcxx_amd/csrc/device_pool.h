// Device memory kept between its owners.
#ifndef DFTGRID_DEVICE_POOL_H
#define DFTGRID_DEVICE_POOL_H

#include <cstddef>
#include <list>
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
// a program that closes many small handles paid for each of them on every allocation),
// and a block that changes hands takes its record along, without the host's allocator
// (a handle of 80 blocks: 6 us, 14 with records made anew).
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
        *p = it->second;
        Block& b = blocks_.find(*p)->second;
        held_ -= it->first.second;
        b.node = kept_.extract(it);
        used_.splice(used_.end(), ages_, b.age);
        return 0;
      }
    }
    if (const int e = raw(p, bytes)) return e;
    if (record(*p, Size{dev, bytes})) return 0;
    Api::release(*p);
    *p = nullptr;
    return Api::kNoMemory;
  }

  // For work that is over on every stream.
  void give(void* p) noexcept {
    std::lock_guard<std::mutex> lock(m_);
    const auto it = blocks_.find(p);
    if (it == blocks_.end() || it->second.node.empty()) return;  // not a block in use
    Block& b = it->second;
    const size_t bytes = b.node.key().second;
    if (bytes > most_) {
      used_.erase(b.age);
      blocks_.erase(it);
      Api::release(p);
      return;
    }
    while (held_ + bytes > most_) drop_oldest();
    b.kept = kept_.insert(std::move(b.node));
    ages_.splice(ages_.end(), used_, b.age);
    held_ += bytes;
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
    const bool any = !ages_.empty();
    while (!ages_.empty()) drop_oldest();
    return any;
  }

 private:
  using Size = std::pair<int, size_t>;  // device, bytes
  using Kept = std::multimap<Size, void*>;
  struct Block {
    typename Kept::node_type node;  // while in use
    typename Kept::iterator kept;   // while kept
    std::list<void*>::iterator age;
  };

  bool record(void* p, Size s) noexcept {
    try {
      Kept one;
      one.emplace(s, p);
      std::lock_guard<std::mutex> lock(m_);
      std::list<void*> age(1, p);
      Block& b = blocks_[p];
      b.node = one.extract(one.begin());
      b.age = age.begin();
      used_.splice(used_.end(), age);
      return true;
    } catch (...) {
      return false;
    }
  }
  void drop_oldest() noexcept {
    void* p = ages_.front();
    const auto it = blocks_.find(p);
    held_ -= it->second.kept->first.second;
    kept_.erase(it->second.kept);
    ages_.pop_front();
    blocks_.erase(it);
    Api::release(p);
  }

  const size_t most_;
  std::mutex m_;
  Kept kept_;
  std::list<void*> ages_, used_;  // kept blocks, oldest first; the others
  std::unordered_map<void*, Block> blocks_;
  size_t held_ = 0;
};

}  // namespace dg

#endif
