// What SitePool takes from the device against what it was asked for: blocks of site sizes, those just above a power of
// two among them, fill their slabs up to a piece smaller than a block, whether of one size or mixed.
#include "../../tnqvm_amd/csrc/site_pool.h"

#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

namespace {
size_t live = 0;
std::unordered_map<void*, size_t> sizes;
struct Heap {
  static void* alloc(size_t n) {
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
using Pool = hipmps::SitePool<Heap>;

size_t site(size_t cl, size_t cr, size_t es) { return cl * 2 * cr * es; }

bool fill(const std::vector<size_t>& kinds, const char* name) {
  Pool pool;
  std::mt19937_64 rng(3);
  size_t asked = 0, count = 0;
  std::vector<void*> blocks;
  while (asked < (size_t)256 << 20) {
    const size_t n = kinds[rng() % kinds.size()];
    blocks.push_back(pool.get(n));
    asked += n;
    ++count;
  }
  // every slab but the last lost less than the block that did not fit any more, and a block less than a grain
  const size_t slabs = live / Pool::SLAB, bound = asked + count * Pool::GRAIN + slabs * Pool::MAX_BLOCK + Pool::SLAB;
  std::printf("%s: %zu MiB asked, %zu MiB held\n", name, asked >> 20, live >> 20);
  if (live > bound) return std::printf("more than %zu MiB\n", bound >> 20), false;
  for (void* p : blocks) pool.put(p);
  return live <= Pool::KEEP_FREE * Pool::SLAB;
}
}  // namespace

int main() {
  const bool ok = fill({site(130, 130, 16)}, "130 x 130") && fill({site(260, 260, 8)}, "260 x 260 complex64") &&
                  fill({site(182, 182, 16)}, "182 x 182") && fill({site(16, 33, 16)}, "16 x 33") &&
                  fill({site(64, 65, 16), site(65, 129, 16), site(130, 200, 16), site(9, 17, 8), 32}, "mixed");
  std::puts(ok && live == 0 ? "ok" : "failed");
  return !(ok && live == 0);
}
