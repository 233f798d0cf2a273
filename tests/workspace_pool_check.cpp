// Drives workspacePool with a device of its own: "memory" is host memory under a budget,
// and every buffer must be freed exactly once.
#include "workspace_pool.hpp"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <memory>
#include <thread>

using libp::workspacePool;

static std::mutex m;
static std::map<void*, size_t> live;
static size_t used = 0, budget = ~size_t(0);

static void* deviceTry(size_t bytes) {
  std::lock_guard<std::mutex> lock(m);
  if (used + bytes > budget) return nullptr;
  void* p = std::malloc(1);
  live[p] = bytes;
  used += bytes;
  return p;
}
static void deviceFree(void* p) {
  std::lock_guard<std::mutex> lock(m);
  auto it = live.find(p);
  if (it == live.end()) {
    std::printf("FAIL: freed twice or never allocated\n");
    std::exit(1);
  }
  used -= it->second;
  live.erase(it);
  std::free(p);
}
static void* deviceAlloc(size_t bytes) {
  return workspacePool::allocate([&] { return deviceTry(bytes); });
}
static void* workspace(workspacePool& pool, size_t bytes) {
  void* p = pool.take(bytes);
  return p ? p : deviceAlloc(bytes);
}
static void expect(bool ok, const char* what) {
  if (!ok) {
    std::printf("FAIL: %s\n", what);
    std::exit(1);
  }
}

int main() {
  {  // the last buffer given of a size comes back, no other size
    workspacePool pool(deviceFree);
    void *a = workspace(pool, 8), *b = workspace(pool, 8);
    pool.give(a, 8);
    pool.give(b, 8);
    expect(pool.take(16) == nullptr, "another size");
    expect(pool.take(8) == b && pool.take(8) == a && pool.take(8) == nullptr, "last given first");
    deviceFree(a);
    pool.give(b, 8);
  }
  expect(used == 0, "freed with the pool");
  {  // at most MOST buffers wait, the oldest are freed
    workspacePool pool(deviceFree);
    void* p[workspacePool::MOST + 5];
    for (size_t i = 0; i < workspacePool::MOST + 5; ++i) p[i] = workspace(pool, 100 + i);
    for (size_t i = 0; i < workspacePool::MOST + 5; ++i) pool.give(p[i], 100 + i);
    expect(live.size() == workspacePool::MOST, "count");
    for (size_t i = 0; i < 5; ++i) expect(pool.take(100 + i) == nullptr, "oldest freed");
    for (size_t i = 5; i < workspacePool::MOST + 5; ++i) {
      expect(pool.take(100 + i) == p[i], "newest kept");
      deviceFree(p[i]);
    }
  }
  expect(used == 0, "freed with the pool (2)");
  {  // at most MOST_BYTES wait; a buffer above them is freed and leaves the others
    workspacePool pool(deviceFree);
    const size_t part = workspacePool::MOST_BYTES / 5 * 2;  // two fit
    void* p[4];
    for (void*& q : p) q = workspace(pool, part);
    void* big = workspace(pool, workspacePool::MOST_BYTES + 1);
    for (void* q : p) pool.give(q, part);
    expect(used - (workspacePool::MOST_BYTES + 1) == 2 * part, "bytes");
    pool.give(big, workspacePool::MOST_BYTES + 1);
    expect(used == 2 * part && pool.take(part) == p[3], "above the limit");
    pool.give(p[3], part);
    void* whole = workspace(pool, workspacePool::MOST_BYTES);
    pool.give(whole, workspacePool::MOST_BYTES);
    expect(used == workspacePool::MOST_BYTES, "a buffer of the limit displaces the others");
  }
  expect(used == 0, "freed with the pool (3)");
  {  // no memory: what waits anywhere is freed, and the allocation succeeds
    budget = 1000;
    workspacePool first(deviceFree), second(deviceFree);
    void *a = workspace(first, 300), *b = workspace(second, 300), *c = workspace(second, 300);
    first.give(a, 300);
    second.give(b, 300);
    void* d = workspace(second, 700);
    expect(d && used == 1000, "another pool's buffers make room");
    expect(workspace(first, 300) == nullptr && deviceAlloc(1) == nullptr, "no room at all");
    second.give(c, 300);
    second.give(d, 700);
    expect(second.drain() == 2 && used == 0 && second.drain() == 0, "drain");
    budget = ~size_t(0);
  }
  {  // a buffer outlives its pool (platform_t::workspaceBytes frees it then), pools come and go
    auto pool = std::make_shared<workspacePool>(deviceFree);
    std::weak_ptr<workspacePool> home = pool;
    void* a = workspace(*pool, 8);
    pool.reset();
    expect(home.expired() && used == 8, "the buffer is its holder's");
    deviceFree(a);
  }
  {  // threads on two shared pools, short of memory most of the time
    budget = 40 * 64;
    workspacePool pools[2] = {workspacePool(deviceFree), workspacePool(deviceFree)};
    std::atomic<int> got{0};
    std::thread t[4];
    for (int k = 0; k < 4; ++k)
      t[k] = std::thread([&, k] {
        unsigned r = 17u + k;
        for (int i = 0; i < 20000; ++i) {
          r = r * 1664525u + 1013904223u;
          const size_t bytes = 64 * (1 + (r >> 8) % 12);
          workspacePool& pool = pools[(r >> 20) & 1];
          if (void* p = workspace(pool, bytes)) {
            ++got;
            pool.give(p, bytes);
          }
          if (i % 100 == 0) {  // a pool that lives for a moment
            workspacePool brief(deviceFree);
            if (void* p = workspace(brief, 64)) brief.give(p, 64);
          }
        }
      });
    for (auto& x : t) x.join();
    expect(got > 40000 && used <= budget, "threads");
  }
  expect(used == 0 && live.empty(), "everything freed");
  std::printf("POOL CHECK OK\n");
  return 0;
}
