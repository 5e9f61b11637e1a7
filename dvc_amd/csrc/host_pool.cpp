// host_pool.cpp -- a context's host copy threads and its pinned staging.
#include <string.h>
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>
#include "dvc_internal.h"

namespace dvc {

// Workers sleep on a condition variable between calls; a call hands out the
// indices 0..count-1 of one job and returns when all are done.  Used by the one
// host thread that holds the context.
struct HostPool {
  std::mutex mu;
  std::condition_variable wake, idle;
  std::vector<std::thread> threads;
  const std::function<void(size_t)> *job = nullptr;
  size_t count = 0;
  std::atomic<size_t> next{0};
  int running = 0;           // workers that have not finished the current job
  unsigned long generation = 0;
  bool stop = false;

  void drain() {
    for (size_t i; (i = next.fetch_add(1)) < count;) (*job)(i);
  }
  void worker() {
    unsigned long seen = 0;
    std::unique_lock<std::mutex> lock(mu);
    for (;;) {
      wake.wait(lock, [&] { return stop || generation != seen; });
      if (stop) return;
      seen = generation;
      lock.unlock();
      drain();
      lock.lock();
      if (--running == 0) idle.notify_one();
    }
  }
  explicit HostPool(int n) {
    try {
      for (int i = 0; i < n; i++) threads.emplace_back([this] { worker(); });
    } catch (...) {  // fewer threads than asked for: the caller's thread does the rest
    }
  }
  ~HostPool() {
    {
      std::lock_guard<std::mutex> lock(mu);
      stop = true;
    }
    wake.notify_all();
    for (auto &t : threads) t.join();
  }
  void run(size_t n, const std::function<void(size_t)> &fn) {
    {
      std::lock_guard<std::mutex> lock(mu);
      job = &fn;
      count = n;
      next = 0;
      running = (int)threads.size();
      generation++;
    }
    wake.notify_all();
    drain();
    std::unique_lock<std::mutex> lock(mu);
    idle.wait(lock, [&] { return running == 0; });
  }
};

void host_pool_free(dvc_ctx *c) {
  delete c->pool;
  c->pool = nullptr;
}

// fn(0..n-1), on the context's threads when `bytes`, the memory it moves, is
// worth waking them (a worker takes some 10 us to start; one thread moves 5 to
// 10 KB in a microsecond, a quarter of that into pages touched for the first
// time).
void host_parallel(dvc_ctx *c, size_t n, size_t bytes, const std::function<void(size_t)> &fn) {
  constexpr int kWorkers = 7;
  if (bytes < (256u << 10) || n < 2) {
    for (size_t i = 0; i < n; i++) fn(i);
    return;
  }
  if (!c->pool) {
    const int cores = (int)std::thread::hardware_concurrency();
    c->pool = new HostPool(std::max(0, std::min(kWorkers, cores - 1)));
  }
  c->pool->run(n, fn);
}

void host_copy(dvc_ctx *c, const std::vector<HostCopy> &list) {
  constexpr size_t kPiece = 128u << 10;
  std::vector<HostCopy> pieces;
  size_t total = 0;
  for (const HostCopy &h : list) {
    total += h.bytes;
    for (size_t o = 0; o < h.bytes; o += kPiece)
      pieces.push_back(HostCopy{(uint8_t *)h.dst + o, (const uint8_t *)h.src + o, std::min(kPiece, h.bytes - o)});
  }
  host_parallel(c, pieces.size(), total, [&](size_t i) { memcpy(pieces[i].dst, pieces[i].src, pieces[i].bytes); });
}

int pinned_grow(uint8_t **p, size_t *have, size_t bytes) {
  if (*have >= bytes) return DVC_OK;
  if (*p) DVC_HIP(hipHostFree(*p));
  *p = nullptr;
  *have = 0;
  DVC_HIP(hipHostMalloc((void **)p, bytes, hipHostMallocDefault));
  *have = bytes;
  return DVC_OK;
}

int copy_back(dvc_ctx *c, hipStream_t s, void *user, const void *dev, uint8_t *pinned, size_t bytes) {
  constexpr size_t kLeast = 1u << 20;
  constexpr int kChunks = 8;
  const size_t chunk = std::max(kLeast, ((bytes + kChunks - 1) / kChunks + 255) & ~(size_t)255);
  hipEvent_t ev[kChunks] = {};
  auto run = [&]() -> int {
    int n = 0;
    for (size_t o = 0; o < bytes; o += chunk, n++) {
      DVC_HIP(hipMemcpyAsync(pinned + o, (const uint8_t *)dev + o, std::min(chunk, bytes - o), hipMemcpyDeviceToHost, s));
      if (o + chunk >= bytes) break;  // the last piece: the stream itself is waited for
      DVC_HIP(hipEventCreateWithFlags(&ev[n], hipEventDisableTiming));
      DVC_HIP(hipEventRecord(ev[n], s));
    }
    int k = 0;
    for (size_t o = 0; o < bytes; o += chunk, k++) {
      if (o + chunk >= bytes) DVC_HIP(hipStreamSynchronize(s));
      else DVC_HIP(hipEventSynchronize(ev[k]));
      host_copy(c, {HostCopy{(uint8_t *)user + o, pinned + o, std::min(chunk, bytes - o)}});
    }
    return DVC_OK;
  };
  const int rc = run();
  for (hipEvent_t e : ev)
    if (e) (void)hipEventDestroy(e);
  return rc;
}

}  // namespace dvc
