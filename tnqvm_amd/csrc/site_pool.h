// site_pool.h -- buddy allocator for the site buffers of an engine (internal).
//
// A bond that grows gives its two sites new buffers and frees the old ones, and a circuit is a few hundred
// such pairs: one hipMalloc and one hipFree each took 7 to 8 us with several circuits in flight (a noisy
// batch of 16 x 40 qubits spent 43 of 98 ms in them, an uneven batch of 32 circuits 90 of 2 x 188 ms on two
// threads).  Blocks up to MAX_BLOCK come from slabs of SLAB bytes by powers of two, the usual ratio of a
// bond's growth, and coalesce with their buddies when freed; larger ones are rare and go to the device
// allocator.  At most KEEP_FREE unused slabs are kept, the others are given back at once.
//
// A block may be handed out again while work that used it is queued: every use of an engine's sites is on
// its stream or on a stream that is ordered with it by events.
#pragma once
#include <cstddef>
#include <iterator>
#include <mutex>
#include <set>
#include <unordered_map>

namespace hipmps {

template <typename Device>  // static void* alloc(size_t) (null on failure), static void free(void*)
class SitePool {
 public:
  static constexpr int MIN_ORDER = 8, MAX_ORDER = 21, SLAB_ORDER = 24;
  static constexpr size_t MAX_BLOCK = (size_t)1 << MAX_ORDER, SLAB = (size_t)1 << SLAB_ORDER;
  static constexpr int KEEP_FREE = 2;

  SitePool() = default;
  SitePool(const SitePool&) = delete;
  ~SitePool() { release(); }

  void* get(size_t bytes) {
    std::lock_guard<std::mutex> lock(mu_);
    if (bytes > MAX_BLOCK) return direct(bytes);
    int want = MIN_ORDER;
    while (((size_t)1 << want) < bytes) ++want;
    int order = want;
    while (order <= SLAB_ORDER && free_[order].empty()) ++order;
    if (order > SLAB_ORDER) {
      char* slab = (char*)Device::alloc(SLAB);
      if (!slab) return direct(bytes);
      slabs_.insert(slab);
      order = SLAB_ORDER;
      free_[order].insert(slab);
    }
    char* p = *free_[order].begin();
    free_[order].erase(free_[order].begin());
    while (order > want) {
      --order;
      free_[order].insert(p + ((size_t)1 << order));
    }
    order_[p] = want;
    return p;
  }

  void put(void* q) {
    if (!q) return;
    std::lock_guard<std::mutex> lock(mu_);
    const auto it = order_.find((char*)q);
    if (it == order_.end()) {
      Device::free(q);
      return;
    }
    char* p = it->first;
    int order = it->second;
    order_.erase(it);
    char* slab = *std::prev(slabs_.upper_bound(p));
    while (order < SLAB_ORDER) {
      char* buddy = slab + ((size_t)(p - slab) ^ ((size_t)1 << order));
      const auto b = free_[order].find(buddy);
      if (b == free_[order].end()) break;
      free_[order].erase(b);
      if (buddy < p) p = buddy;
      ++order;
    }
    if (order == SLAB_ORDER && free_[order].size() >= KEEP_FREE) {
      slabs_.erase(p);
      Device::free(p);
    } else {
      free_[order].insert(p);
    }
  }

  void release() {
    std::lock_guard<std::mutex> lock(mu_);
    for (char* s : slabs_) Device::free(s);
    slabs_.clear();
    order_.clear();
    for (auto& f : free_) f.clear();
  }

 private:
  // the device allocator, once more without the slabs kept free
  void* direct(size_t bytes) {
    void* p = Device::alloc(bytes);
    if (p || free_[SLAB_ORDER].empty()) return p;
    for (char* s : free_[SLAB_ORDER]) {
      slabs_.erase(s);
      Device::free(s);
    }
    free_[SLAB_ORDER].clear();
    return Device::alloc(bytes);
  }

  std::mutex mu_;
  std::set<char*> slabs_;
  std::set<char*> free_[SLAB_ORDER + 1];
  std::unordered_map<char*, int> order_;  // of the blocks handed out
};

}  // namespace hipmps
