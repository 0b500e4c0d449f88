// Device blocks of freed meshes, kept for the next mesh (host code, no HIP in
// it: the function that frees a block is given).
//
// A mesh is built, read and freed again and again (a surface per time step),
// and at 256^3 and two thresholds the driver took 42 ms to allocate and free
// what the kernels fill in 1.3 ms.  At most `limit` bytes are held; the oldest
// blocks go first.  A block may come here only once the device is done with
// it, so that any stream may take it, and only of the device that the library
// is initialised on, which all blocks of a pool belong to.
#pragma once

#include <cstddef>
#include <mutex>
#include <vector>

namespace c3d {

struct BlockPool {
  struct Block {
    void* p;
    size_t bytes;
  };
  const size_t limit;
  void (*const free_block)(void*);
  std::mutex mu;
  std::vector<Block> blocks;  // oldest first
  size_t held = 0;
  BlockPool(size_t limit_, void (*free_block_)(void*)) : limit(limit_), free_block(free_block_) {}
  // the smallest block of at least `want` bytes that is not more than twice
  // that (small requests: 64 KiB more)
  void* take(size_t want, size_t& got) {
    std::lock_guard<std::mutex> g(mu);
    size_t best = blocks.size();
    for (size_t q = 0; q < blocks.size(); q++)
      if (blocks[q].bytes >= want && blocks[q].bytes <= 2 * want + 65536 &&
          (best == blocks.size() || blocks[q].bytes < blocks[best].bytes))
        best = q;
    if (best == blocks.size()) return nullptr;
    void* p = blocks[best].p;
    got = blocks[best].bytes;
    held -= got;
    blocks.erase(blocks.begin() + std::ptrdiff_t(best));
    return p;
  }
  void give(void* p, size_t bytes) {
    std::lock_guard<std::mutex> g(mu);
    if (bytes > limit) {
      free_block(p);
      return;
    }
    while (held + bytes > limit) {
      held -= blocks.front().bytes;
      free_block(blocks.front().p);
      blocks.erase(blocks.begin());
    }
    blocks.push_back({p, bytes});
    held += bytes;
  }
  // frees every block; false if there was none
  bool drop() {
    std::lock_guard<std::mutex> g(mu);
    const bool any = !blocks.empty();
    for (const Block& b : blocks) free_block(b.p);
    blocks.clear();
    held = 0;
    return any;
  }
};

}  // namespace c3d
