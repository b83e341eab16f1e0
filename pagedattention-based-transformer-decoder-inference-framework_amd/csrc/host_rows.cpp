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
};

struct Pool {
  static constexpr size_t kMost = (size_t)64 << 20;     // all blocks, lent or free
  static constexpr size_t kAhead = (size_t)8 << 20;     // a block made with an engine
  static constexpr size_t kUnit = (size_t)256 << 10;
  std::mutex mu;
  std::vector<Block> blocks;
  size_t total = 0;
  int engines = 0;

  // Free blocks of up to 4 times the size, so that small results do not hold large blocks.
  Block* find(size_t bytes) {
    Block* best = nullptr;
    for (Block& b : blocks)
      if (!b.lent && b.size >= bytes && b.size <= 4 * bytes + kUnit && (!best || b.size < best->size)) best = &b;
    return best;
  }
  void drop(size_t i) {
    (void)hipHostFree(blocks[i].p);
    total -= blocks[i].size;
    blocks.erase(blocks.begin() + i);
  }
  Block* make(size_t bytes) {
    const size_t size = (bytes + kUnit - 1) / kUnit * kUnit;
    for (size_t i = blocks.size(); i-- > 0 && total + size > kMost;)
      if (!blocks[i].lent) drop(i);
    if (total + size > kMost) return nullptr;
    Block b;
    if (hipHostMalloc(reinterpret_cast<void**>(&b.p), size, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    b.size = size;
    total += size;
    blocks.push_back(b);
    return &blocks.back();
  }
};
Pool& pool() {
  static Pool* p = new Pool();  // arrays may outlive the library's static objects
  return *p;
}

}  // namespace

// Two blocks: a caller holds one step's rows while the next one runs.  The host's first touch
// of a page costs 1.5 us.
void host_rows_engine_begins(size_t bytes) {
  Pool& p = pool();
  std::lock_guard<std::mutex> g(p.mu);
  ++p.engines;
  if (bytes > Pool::kAhead) return;
  int ready = 0;
  for (const Block& b : p.blocks) ready += !b.lent && b.size >= bytes && b.size <= 4 * bytes + Pool::kUnit;
  for (; ready < 2; ++ready) {
    Block* b = p.make(bytes);
    if (!b) return;
    std::memset(b->p, 0, b->size);
  }
}

void host_rows_engine_ends() {
  Pool& p = pool();
  std::lock_guard<std::mutex> g(p.mu);
  if (--p.engines > 0) return;
  for (size_t i = p.blocks.size(); i-- > 0;)
    if (!p.blocks[i].lent) p.drop(i);
}

}  // namespace llm

using namespace llm;

extern "C" void* llm_host_rows_take(size_t bytes) {
  Pool& p = pool();
  std::lock_guard<std::mutex> g(p.mu);
  if (p.engines == 0 || bytes == 0) return nullptr;
  Block* b = p.find(bytes);
  if (!b) b = p.make(bytes);
  if (!b) return nullptr;
  b->lent = true;
  return b->p;
}

extern "C" void llm_host_rows_give(void* at) {
  Pool& p = pool();
  std::lock_guard<std::mutex> g(p.mu);
  for (size_t i = 0; i < p.blocks.size(); ++i)
    if (p.blocks[i].p == at && p.blocks[i].lent) {
      p.blocks[i].lent = false;
      if (p.engines == 0) p.drop(i);
      return;
    }
}
