// Host check of c3d_pool.h against a model: random blocks given and taken
// through a pool of a small limit.  What is held never exceeds the limit and
// is exactly what was given, not taken and not freed; the oldest block is the
// first to be freed; a block taken fits (the smallest that does); a block
// larger than the limit is freed at once; drop frees the rest.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>

#include "c3d_pool.h"

static std::vector<void*> freed;
static void free_block(void* p) { freed.push_back(p); }
static void check(bool ok, const char* what) {
  if (ok) return;
  std::printf("FAILED: %s\n", what);
  std::exit(1);
}

int main() {
  const size_t limit = 1 << 20;
  c3d::BlockPool pool(limit, free_block);
  check(!pool.drop(), "an empty pool has nothing to drop");
  std::mt19937 g(3);
  std::vector<std::pair<void*, size_t>> model;  // oldest first
  uintptr_t next = 16;
  size_t evicted = 0, taken = 0, missed = 0, dropped = 0;
  for (int step = 0; step < 20000; step++) {
    const size_t n = 1 + g() % (g() % 8 ? 150000 : limit + 5000);
    if (g() % 2) {
      void* p = reinterpret_cast<void*>(next += 16);
      freed.clear();
      pool.give(p, n);
      if (n > limit) {
        check(freed.size() == 1 && freed[0] == p, "a block over the limit is freed at once");
        continue;
      }
      for (void* f : freed) {
        check(f == model.front().first, "the oldest goes first");
        model.erase(model.begin());
        evicted++;
      }
      model.push_back({p, n});
    } else {
      size_t got = 0, best = model.size();
      for (size_t q = 0; q < model.size(); q++)
        if (model[q].second >= n && model[q].second <= 2 * n + 65536 &&
            (best == model.size() || model[q].second < model[best].second))
          best = q;
      void* p = pool.take(n, got);
      if (best == model.size()) {
        check(!p, "no block fits");
        missed++;
      } else {
        check(p == model[best].first && got == model[best].second, "the smallest that fits");
        model.erase(model.begin() + std::ptrdiff_t(best));
        taken++;
      }
    }
    size_t sum = 0;
    for (const auto& b : model) sum += b.second;
    check(pool.held == sum && sum <= limit && pool.blocks.size() == model.size(), "held bytes");
    if (g() % 500 == 0) {
      freed.clear();
      check(pool.drop() == !model.empty() && freed.size() == model.size() && pool.held == 0, "drop frees all");
      dropped += freed.size();
      model.clear();
    }
  }
  check(evicted > 100 && taken > 100 && missed > 100 && dropped > 10, "every path was taken");
  std::printf("ok: %zu taken, %zu missed, %zu evicted, %zu dropped\n", taken, missed, evicted, dropped);
  return 0;
}
