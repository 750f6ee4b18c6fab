#include "ps_pool.hpp"

#include <map>
#include <mutex>
#include <vector>

#include "../../include/partapp_ps.h"
#include "ps_plan.hpp"

namespace ps {

namespace {

struct Block {
  void *p;
  size_t bytes;
  int dev;
};

// never destroyed: a plan may outlive the library's static objects
struct Pool {
  std::mutex mu;
  std::vector<Block> idle;          // oldest first
  std::map<void *, Block> lent;
  std::vector<unsigned *> words;    // idle
};
Pool &pool() {
  static Pool *p = new Pool;
  return *p;
}

// the cached blocks of a device, taken out of the pool (freed by the caller,
// outside the lock)
std::vector<Block> take_idle(Pool &q, int dev) {
  std::vector<Block> out, keep;
  for (const Block &b : q.idle) (b.dev == dev ? out : keep).push_back(b);
  q.idle.swap(keep);
  return out;
}

}  // namespace

hipError_t pool_get(void **p, size_t bytes) {
  *p = nullptr;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (bytes == 0) bytes = 1;
  Pool &q = pool();
  {
    // the tightest block that wastes at most a quarter (or 1 MiB)
    std::lock_guard<std::mutex> lock(q.mu);
    size_t best = q.idle.size();
    for (size_t i = 0; i < q.idle.size(); ++i) {
      const Block &b = q.idle[i];
      if (b.dev == dev && b.bytes >= bytes && b.bytes <= bytes + bytes / 4 + (1u << 20) &&
          (best == q.idle.size() || b.bytes < q.idle[best].bytes))
        best = i;
    }
    if (best < q.idle.size()) {
      const Block b = q.idle[best];
      q.idle.erase(q.idle.begin() + (long)best);
      q.lent[b.p] = b;
      *p = b.p;
      return hipSuccess;
    }
  }
  e = hipMalloc(p, bytes);
  if (e != hipSuccess) {
    std::vector<Block> freed;
    {
      std::lock_guard<std::mutex> lock(q.mu);
      freed = take_idle(q, dev);
    }
    if (freed.empty()) return e;
    (void)hipGetLastError();
    for (const Block &b : freed) (void)hipFree(b.p);
    e = hipMalloc(p, bytes);
    if (e != hipSuccess) return e;
  }
  std::lock_guard<std::mutex> lock(q.mu);
  q.lent[*p] = Block{*p, bytes, dev};
  return hipSuccess;
}

void pool_put(void *p, bool idle) {
  if (!p) return;
  Pool &q = pool();
  std::vector<Block> freed;
  {
    std::lock_guard<std::mutex> lock(q.mu);
    auto it = q.lent.find(p);
    const Block b = it != q.lent.end() ? it->second : Block{p, 0, -1};
    if (it != q.lent.end()) q.lent.erase(it);
    if (!idle || b.dev < 0 || b.bytes > kPoolBytes) {
      freed.push_back(b);
    } else {
      q.idle.push_back(b);
      size_t bytes = 0, n = 0;
      for (const Block &i : q.idle)
        if (i.dev == b.dev) bytes += i.bytes, ++n;
      for (size_t i = 0; i < q.idle.size() && (bytes > kPoolBytes || n > kPoolBlocks);) {
        if (q.idle[i].dev != b.dev) {
          ++i;
          continue;
        }
        bytes -= q.idle[i].bytes;
        --n;
        freed.push_back(q.idle[i]);
        q.idle.erase(q.idle.begin() + (long)i);
      }
    }
  }
  for (const Block &b : freed) (void)hipFree(b.p);
}

hipError_t pool_get_host(unsigned **p) {
  *p = nullptr;
  Pool &q = pool();
  {
    std::lock_guard<std::mutex> lock(q.mu);
    if (!q.words.empty()) {
      *p = q.words.back();
      q.words.pop_back();
      return hipSuccess;
    }
  }
  // portable: any device's kernels write it
  return hipHostMalloc(reinterpret_cast<void **>(p), sizeof(unsigned), hipHostMallocPortable);
}

void pool_put_host(unsigned *p, bool idle) {
  if (!p) return;
  Pool &q = pool();
  if (idle) {
    std::lock_guard<std::mutex> lock(q.mu);
    if (q.words.size() < kPoolWords) {
      q.words.push_back(p);
      return;
    }
  }
  (void)hipHostFree(p);
}

hipError_t pool_trim() {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  Pool &q = pool();
  std::vector<Block> freed;
  std::vector<unsigned *> words;
  {
    std::lock_guard<std::mutex> lock(q.mu);
    freed = take_idle(q, dev);
    words.swap(q.words);
  }
  for (const Block &b : freed) {
    const hipError_t f = hipFree(b.p);
    if (e == hipSuccess) e = f;
  }
  for (unsigned *w : words) {
    const hipError_t f = hipHostFree(w);
    if (e == hipSuccess) e = f;
  }
  return e;
}

}  // namespace ps

extern "C" int ps_release_memory(void) {
  const hipError_t e = ps::pool_trim();
  if (e != hipSuccess) return ps::set_error(PS_ERR_HIP, std::string("releasing memory: ") + hipGetErrorString(e));
  return PS_OK;
}
