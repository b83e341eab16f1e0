// Pinned blocks that a step's logits arrive in and that its caller then holds: one copy over
// the bus, where pageable memory takes the pieces of a ring and a copy out of them into pages
// that the host touches for the first time (64 rows of 32,768: 586 us a step, now 456; 16 rows
// 399, 351).  Blocks come back when the arrays over them go, from any thread; the copies into
// them were waited for by then.
#include "host_rows.hpp"

#include <hip/hip_runtime.h>

#include <cstring>
#include <mutex>
#include <vector>

#include "llm_decoder.h"

namespace llm {
namespace {

struct Block {
  char* p = nullptr;
  size_t size = 0;
  bool lent = false;
  uint64_t used = 0;  // the last take while it was lent
};

struct Pool {
  static constexpr size_t kMost = (size_t)64 << 20;     // all blocks, lent or free
  static constexpr size_t kAhead = (size_t)8 << 20;     // a block made with an engine
  static constexpr size_t kUnit = (size_t)256 << 10;
  // A free block makes room for another after that many takes without it: results of two sizes in
  // turn, which do not both fit, would else free and pin a block at every step (60 MiB: 30 us and 15
  // to 900).  The one without a block takes memory of its own.
  static constexpr uint64_t kIdle = 64;
  std::mutex mu;
  std::vector<Block> blocks;
  size_t total = 0;  // of blocks, and of those being made
  uint64_t takes = 0;
  int engines = 0;

  static bool fits(const Block& b, size_t bytes) {
    // (up to 4 times the size, so that small results do not hold large blocks)
    return !b.lent && b.size >= bytes && b.size <= 4 * bytes + kUnit;
  }
  Block* find(size_t bytes) {
    Block* best = nullptr;
    for (Block& b : blocks)
      if (fits(b, bytes) && (!best || b.size < best->size)) best = &b;
    return best;
  }
  char* remove(size_t i) {
    char* p = blocks[i].p;
    total -= blocks[i].size;
    blocks.erase(blocks.begin() + i);
    return p;
  }
  bool idle(const Block& b) const { return !b.lent && takes - b.used >= kIdle; }
  // A new block; null: there is no room or none to pin.  `mu` is not held while memory is pinned or
  // given back, so that nobody's take or give waits for it.
  char* make(size_t bytes, bool lent, std::unique_lock<std::mutex>& lock) {
    const size_t size = (bytes + kUnit - 1) / kUnit * kUnit;
    size_t free = 0;
    for (const Block& b : blocks) free += idle(b) ? b.size : 0;
    if (total - free + size > kMost) return nullptr;
    std::vector<char*> out;
    while (total + size > kMost) {
      size_t oldest = blocks.size();
      for (size_t i = 0; i < blocks.size(); ++i)
        if (idle(blocks[i]) && (oldest == blocks.size() || blocks[i].used < blocks[oldest].used)) oldest = i;
      out.push_back(remove(oldest));
    }
    total += size;
    lock.unlock();
    for (char* p : out) (void)hipHostFree(p);
    void* p = nullptr;
    if (hipHostMalloc(&p, size, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      p = nullptr;
    }
    if (p && !lent) std::memset(p, 0, size);  // the host's first touch of a page costs 1.5 us
    lock.lock();
    if (!p) {
      total -= size;
      return nullptr;
    }
    blocks.push_back({static_cast<char*>(p), size, lent, takes});
    return static_cast<char*>(p);
  }
};
Pool& pool() {
  static Pool* p = new Pool();  // arrays may outlive the library's static objects
  return *p;
}

}  // namespace

// Two blocks: a caller holds one step's rows while the next one runs.
void host_rows_engine_begins(size_t bytes) {
  Pool& p = pool();
  std::unique_lock<std::mutex> lock(p.mu);
  ++p.engines;
  if (bytes > Pool::kAhead) return;
  int ready = 0;
  for (const Block& b : p.blocks) ready += Pool::fits(b, bytes);
  for (; ready < 2; ++ready)
    if (!p.make(bytes, false, lock)) return;
}

void host_rows_engine_ends() {
  Pool& p = pool();
  std::vector<char*> out;
  {
    std::lock_guard<std::mutex> g(p.mu);
    if (--p.engines > 0) return;
    for (size_t i = p.blocks.size(); i-- > 0;)
      if (!p.blocks[i].lent) out.push_back(p.remove(i));
  }
  for (char* b : out) (void)hipHostFree(b);
}

}  // namespace llm

using namespace llm;

extern "C" void* llm_host_rows_take(size_t bytes) {
  Pool& p = pool();
  std::unique_lock<std::mutex> lock(p.mu);
  if (p.engines == 0 || bytes == 0 || bytes > Pool::kMost) return nullptr;
  ++p.takes;
  if (Block* b = p.find(bytes)) {
    b->lent = true;
    b->used = p.takes;
    return b->p;
  }
  return p.make(bytes, true, lock);
}

extern "C" size_t llm_host_rows_held(const void* at) {
  Pool& p = pool();
  std::lock_guard<std::mutex> g(p.mu);
  for (const Block& b : p.blocks)
    if (b.p == at && b.lent) return b.size;
  return 0;
}

extern "C" void llm_host_rows_give(void* at) {
  Pool& p = pool();
  {
    std::lock_guard<std::mutex> g(p.mu);
    size_t i = 0;
    while (i < p.blocks.size() && !(p.blocks[i].p == at && p.blocks[i].lent)) ++i;
    if (i == p.blocks.size()) return;
    p.blocks[i].lent = false;
    p.blocks[i].used = p.takes;
    if (p.engines > 0) return;
    (void)p.remove(i);
  }
  (void)hipHostFree(at);
}
