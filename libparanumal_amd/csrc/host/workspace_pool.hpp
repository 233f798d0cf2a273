/* Device buffers that wait for the next caller of their size
 * (platform_t::workspace). What waits is memory that nothing else can use, so
 * it is bounded by count and by bytes (the oldest are freed first), and every
 * pool of the process is emptied when an allocation fails. Freeing is passed
 * in, so that this file knows no device. Any thread may call anything here. */
#pragma once

#include <cstddef>
#include <mutex>
#include <utility>
#include <vector>

namespace libp {

class workspacePool {
 public:
  // The vectors of a 32^3, N = 7 solve (16.8M nodes) fit: with half of this its p-MG run took
  // 21.1 ms and not 19.7. From there on allocating is a small share of a solve (40^3: 2.0 GB
  // would wait, and 6.1 ms beside the iterations become 7.7).
  static constexpr size_t MOST = 16, MOST_BYTES = size_t(1) << 30;
  using release_t = void (*)(void*);

  explicit workspacePool(release_t release_) : release(release_) {
    waiting.reserve(MOST + 1);  // give() does not allocate: it runs where nothing may be thrown
    std::lock_guard<std::mutex> lock(all().m);
    all().pools.push_back(this);
  }
  workspacePool(const workspacePool&) = delete;
  workspacePool& operator=(const workspacePool&) = delete;
  ~workspacePool() {
    {
      std::lock_guard<std::mutex> lock(all().m);
      for (auto& p : all().pools)
        if (p == this) {
          std::swap(p, all().pools.back());
          all().pools.pop_back();
          break;
        }
    }
    drain();
  }

  // The buffer of this size that was given last, or null.
  void* take(size_t bytes) {
    std::lock_guard<std::mutex> lock(m);
    for (size_t i = waiting.size(); i-- > 0;)
      if (waiting[i].first == bytes) {
        void* p = waiting[i].second;
        waiting.erase(waiting.begin() + i);
        held -= bytes;
        return p;
      }
    return nullptr;
  }

  void give(void* p, size_t bytes) noexcept {
    if (bytes > MOST_BYTES) return release(p);
    void* old[MOST + 1];
    size_t n = 0;
    {
      std::lock_guard<std::mutex> lock(m);
      waiting.emplace_back(bytes, p);
      held += bytes;
      for (; waiting.size() - n > MOST || held > MOST_BYTES; ++n) {
        held -= waiting[n].first;
        old[n] = waiting[n].second;
      }
      waiting.erase(waiting.begin(), waiting.begin() + n);
    }
    for (size_t i = 0; i < n; ++i) release(old[i]);
  }

  // Frees what waits; the number of buffers freed.
  size_t drain() noexcept {
    void* old[MOST];
    size_t n = 0;
    {
      std::lock_guard<std::mutex> lock(m);
      for (auto& w : waiting) old[n++] = w.second;
      waiting.clear();
      held = 0;
    }
    for (size_t i = 0; i < n; ++i) release(old[i]);
    return n;
  }

  // tryAlloc(): a pointer, or null when there is no memory. Every pool is emptied before
  // the one further try: the memory may wait in the pool of another platform.
  template <typename F>
  static void* allocate(F&& tryAlloc) {
    void* p = tryAlloc();
    if (p) return p;
    size_t freed = 0;
    {
      std::lock_guard<std::mutex> lock(all().m);
      for (workspacePool* w : all().pools) freed += w->drain();
    }
    return freed ? tryAlloc() : nullptr;
  }

 private:
  struct registry {
    std::mutex m;
    std::vector<workspacePool*> pools;
  };
  static registry& all() {
    static registry* r = new registry;  // outlives every platform, static ones too
    return *r;
  }
  release_t release;
  std::mutex m;
  size_t held = 0;
  std::vector<std::pair<size_t, void*>> waiting;  // oldest first
};

}  // namespace libp
