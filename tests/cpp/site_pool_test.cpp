// SitePool against malloc: blocks never overlap, hold their bytes until freed, coalesce back to whole slabs,
// and a failing device allocator is answered with null and leaves the pool usable.
#include "../../tnqvm_amd/csrc/site_pool.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

namespace {
size_t live = 0, limit = 0;
std::unordered_map<void*, size_t> sizes;
struct Heap {
  static void* alloc(size_t n) {
    if (live + n > limit) return nullptr;
    void* p = std::malloc(n);
    sizes[p] = n;
    live += n;
    return p;
  }
  static void free(void* p) {
    live -= sizes.at(p);
    sizes.erase(p);
    std::free(p);
  }
};
struct Block {
  unsigned char* p;
  size_t n;
  unsigned char tag;
};
}  // namespace

int main(int argc, char** argv) {
  limit = (size_t)(argc > 1 ? std::atoi(argv[1]) : 1024) << 20;
  using Pool = hipmps::SitePool<Heap>;
  Pool pool;
  std::mt19937_64 rng(7);
  std::vector<Block> blocks;
  int refused = 0;
  for (int k = 0; k < 30000; ++k) {
    const bool grow = rng() % 100 < ((k / 5000) % 2 ? 45u : 55u);
    if (blocks.empty() || grow) {
      size_t n = (size_t)1 << rng() % 23;
      n = n / 2 + rng() % n + 1;
      auto* p = (unsigned char*)pool.get(n);
      if (!p) {
        ++refused;
        continue;
      }
      const unsigned char tag = (unsigned char)rng();
      std::memset(p, tag, n);
      blocks.push_back({p, n, tag});
    } else {
      const size_t i = rng() % blocks.size();
      const Block b = blocks[i];
      for (size_t e = 0; e < b.n; e += b.n < 64 ? 1 : b.n / 61)
        if (b.p[e] != b.tag) return std::puts("a block was overwritten"), 1;
      if (b.p[b.n - 1] != b.tag) return std::puts("a block's end was overwritten"), 1;
      pool.put(b.p);
      blocks[i] = blocks.back();
      blocks.pop_back();
    }
  }
  for (auto& b : blocks) pool.put(b.p);
  if (live > Pool::KEEP_FREE * Pool::SLAB) return std::puts("unused slabs were kept"), 1;
  pool.release();
  if (live) return std::puts("slabs left after release"), 1;
  std::printf("ok, %d refused\n", refused);
  return 0;
}
