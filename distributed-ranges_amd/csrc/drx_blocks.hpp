// drx_blocks.hpp -- device memory that objects take and give back (host code;
// the runtime's calls come from Driver, so that it can be tested without a GPU).
//
// A block on the free list serves any stream at once, so it may go there only
// when no work that uses it is left. Blocks of an object that any stream may
// have used are retired: they wait aside until the device has been waited for.
// The runtime can refuse that wait (while a stream is being captured), and then
// they stay aside until a later one succeeds.
#pragma once

#include <algorithm>
#include <cstddef>
#include <initializer_list>
#include <list>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace drx {

// Driver: static functions of the current device.
//   int alloc(void **p, size_t bytes)  0, kOutOfMemory or another status
//   bool free(void *p)                 false: refused, p is still allocated
//   bool wait()                        true: all work queued before has ended
// At most Keep bytes are kept; sizes are rounded up to a Quantum.
template <typename Driver, size_t Keep, size_t Quantum = 4096> class BlockCache {
public:
  // A block of at least `bytes`, or the status of the failed allocation. A
  // failed one gives all kept blocks back and tries again.
  int take(size_t bytes, void **out) {
    bytes = (std::max<size_t>(bytes, 1) + Quantum - 1) / Quantum * Quantum;
    if (find(bytes, out)) return 0;
    if (settle() && find(bytes, out)) return 0;
    void *p = nullptr;
    int e = Driver::alloc(&p, bytes);
    if (e == Driver::kOutOfMemory && release()) e = Driver::alloc(&p, bytes);
    if (e != 0) return e;
    std::lock_guard<std::mutex> lk(mu_);
    size_[p].bytes = bytes;
    *out = p;
    return 0;
  }

  // A block that no work uses any more.
  void give(void *p) {
    std::lock_guard<std::mutex> lk(mu_);
    keep(p);
    while (total_ > Keep && drop(order_.front())) {
    }
  }

  // Blocks that queued work may still use; whether the device has been waited for.
  template <typename Ptrs> bool retire(const Ptrs &ptrs) {
    {
      std::lock_guard<std::mutex> lk(mu_);
      for (void *p : ptrs)
        if (size_.count(p)) parked_.push_back(p);
    }
    return settle();
  }

  // Waits for the device, and keeps the blocks that were retired before; false
  // when there are none or the wait is refused.
  bool settle() {
    std::vector<void *> had;
    {
      std::lock_guard<std::mutex> lk(mu_);
      had.swap(parked_);
    }
    if (had.empty()) return false;
    const bool waited = Driver::wait();
    std::lock_guard<std::mutex> lk(mu_);
    if (!waited) {
      parked_.insert(parked_.end(), had.begin(), had.end());
      return false;
    }
    for (void *p : had) keep(p);
    while (total_ > Keep && drop(order_.front())) {
    }
    return true;
  }

  // Gives all kept blocks back to the driver; whether there were any.
  bool release() {
    settle();
    std::lock_guard<std::mutex> lk(mu_);
    const size_t had = total_;
    while (!order_.empty() && drop(order_.front())) {
    }
    return total_ < had;
  }

  bool owns(void *p) {
    std::lock_guard<std::mutex> lk(mu_);
    return size_.count(p) != 0;
  }
  // Bytes kept for reuse.
  size_t kept() {
    std::lock_guard<std::mutex> lk(mu_);
    return total_;
  }

private:
  // A kept block of at most a quarter (small ones: 64 KB) more.
  bool find(size_t bytes, void **out) {
    std::lock_guard<std::mutex> lk(mu_);
    const auto it = kept_.lower_bound(bytes);
    if (it == kept_.end() || it->first > bytes + std::max<size_t>(bytes / 4, 65536)) return false;
    *out = it->second;
    forget(size_[it->second]);
    return true;
  }
  void keep(void *p) {
    const auto at = size_.find(p);
    if (at == size_.end()) return;
    Block &b = at->second;
    b.by_size = kept_.emplace(b.bytes, p);
    b.by_age = order_.insert(order_.end(), p);
    total_ += b.bytes;
  }
  // A kept block goes back to the driver; false: refused, it stays.
  bool drop(void *p) {
    if (!Driver::free(p)) return false;
    forget(size_[p]);
    size_.erase(p);
    return true;
  }

  // Out of the kept ones (by iterator: searching the list of hundreds of slots
  // that a closed batch leaves cost 10 us per plan).
  struct Block {
    size_t bytes = 0;
    std::multimap<size_t, void *>::iterator by_size;  // these two: a kept one's
    std::list<void *>::iterator by_age;
  };
  void forget(Block &b) {
    kept_.erase(b.by_size);
    order_.erase(b.by_age);
    total_ -= b.bytes;
  }

  std::mutex mu_;
  std::unordered_map<void *, Block> size_;  // every block handed out, kept or retired
  std::multimap<size_t, void *> kept_;      // by size
  std::list<void *> order_;                 // kept ones, oldest first
  std::vector<void *> parked_;              // retired, not waited for yet
  size_t total_ = 0;                        // bytes kept
};

}  // namespace drx
