// site_pool.h -- allocator for the site buffers of an engine (internal).
//
// A bond that grows gives its two sites new buffers and frees the old ones, and a circuit is a few hundred
// such pairs: one hipMalloc and one hipFree each took 7 to 8 us with several circuits in flight (a noisy
// batch of 16 x 40 qubits spent 43 of 98 ms in them, an uneven batch of 32 circuits 90 of 2 x 188 ms on two
// threads).  Blocks up to MAX_BLOCK come from slabs of SLAB bytes, the smallest free piece that holds them
// cut to GRAIN bytes, so that what the device holds is what the engine's budget counts and at most an eighth
// more at the slabs' ends (powers of two would be up to twice it); free neighbours join again.  Larger ones
// are rare and go to the device allocator.  At most KEEP_FREE unused slabs are kept, the others are given
// back at once.
//
// A block may be handed out again while work that used it is queued: every use of an engine's sites is on
// its stream or on a stream that is ordered with it by events.
#pragma once
#include <cstddef>
#include <iterator>
#include <map>
#include <mutex>
#include <set>
#include <unordered_map>
#include <utility>

namespace hipmps {

template <typename Device>  // static void* alloc(size_t) (null on failure), static void free(void*)
class SitePool {
 public:
  static constexpr size_t GRAIN = 256, MAX_BLOCK = (size_t)2 << 20, SLAB = (size_t)16 << 20;
  static constexpr int KEEP_FREE = 2;

  SitePool() = default;
  SitePool(const SitePool&) = delete;
  ~SitePool() { release(); }

  void* get(size_t bytes) {
    std::lock_guard<std::mutex> lock(mu_);
    if (bytes > MAX_BLOCK) return direct(bytes);
    const size_t want = bytes ? (bytes + GRAIN - 1) / GRAIN * GRAIN : GRAIN;
    auto it = by_size_.lower_bound({want, nullptr});
    if (it == by_size_.end()) {
      char* slab = (char*)Device::alloc(SLAB);
      if (!slab) return direct(bytes);
      slabs_.insert(slab);
      add(slab, SLAB);
      it = by_size_.find({SLAB, slab});
    }
    const auto [size, p] = *it;
    remove(p, size);
    if (size > want) add(p + want, size - want);
    used_[p] = want;
    return p;
  }

  void put(void* q) {
    if (!q) return;
    std::lock_guard<std::mutex> lock(mu_);
    const auto u = used_.find((char*)q);
    if (u == used_.end()) {
      Device::free(q);
      return;
    }
    char* p = u->first;
    size_t size = u->second;
    used_.erase(u);
    char* slab = *std::prev(slabs_.upper_bound(p));  // slabs may be neighbours: pieces join within one
    auto next = free_.lower_bound(p);
    if (next != free_.end() && next->first == p + size && next->first < slab + SLAB) {
      size += next->second;
      remove(next->first, next->second);
    }
    next = free_.lower_bound(p);
    if (next != free_.begin()) {
      const auto before = *std::prev(next);
      if (before.first >= slab && before.first + before.second == p) {
        p = before.first;
        size += before.second;
        remove(before.first, before.second);
      }
    }
    if (size == SLAB && whole_ >= KEEP_FREE) {
      slabs_.erase(p);
      Device::free(p);
    } else {
      add(p, size);
    }
  }

  void release() {
    std::lock_guard<std::mutex> lock(mu_);
    for (char* s : slabs_) Device::free(s);
    slabs_.clear();
    used_.clear();
    free_.clear();
    by_size_.clear();
    whole_ = 0;
  }

 private:
  void add(char* p, size_t size) {
    free_[p] = size;
    by_size_.insert({size, p});
    whole_ += size == SLAB;
  }
  void remove(char* p, size_t size) {
    free_.erase(p);
    by_size_.erase({size, p});
    whole_ -= size == SLAB;
  }
  // the device allocator, once more without the slabs kept free
  void* direct(size_t bytes) {
    void* p = Device::alloc(bytes);
    if (p || whole_ == 0) return p;
    while (whole_ > 0) {
      char* s = by_size_.rbegin()->second;
      remove(s, SLAB);
      slabs_.erase(s);
      Device::free(s);
    }
    return Device::alloc(bytes);
  }

  std::mutex mu_;
  std::set<char*> slabs_;
  std::map<char*, size_t> free_;                   // pieces by address
  std::set<std::pair<size_t, char*>> by_size_;     // and by size
  int whole_ = 0;                                  // free pieces that are whole slabs
  std::unordered_map<char*, size_t> used_;         // blocks handed out
};

}  // namespace hipmps
