// Downloads: device memory to pageable host memory.
//
// The runtime's own copy to pageable memory reaches 10 GB/s (12 MB 1.24 ms, 38 MB
// 3.9 ms, 134 MB 13.6 ms: one host thread copies out of a staging buffer and
// takes the destination's page faults); the link does 53.  Here a kernel writes
// chunks into a ring of pinned memory (the runtime's copy engines cost 6 ms at
// first use) and host threads copy them on in parts of 256 KB: 12 MB 0.40 ms,
// 38 MB 1.2, 134 MB 3.7.  The calling thread issues the chunks and copies parts
// like any other, and no thread takes a part before its chunk has landed, so a
// helper that the host does not schedule holds nothing up.
//
// A chunk is an eighth of the download, at most 2 MB, with four in flight: the
// host's first read of new pinned memory takes 0.37 ms a MB (page faults), so
// the ring of a small download is small (eight slots gain 5 % over four).
// Three helpers up to 24 MB, seven beyond (11 are no faster).
//
// Rings and threads are shared by the contexts of the process.  A download has
// a ring to itself; at most two are kept while none needs them.  The last
// context gives all of it back.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace dl {

constexpr int kSlots = 4;
constexpr size_t kPart = 256u << 10;

struct Ring {
  char* p = nullptr;
  char* d = nullptr;  // as the device sees it
  size_t bytes = 0;
};

struct Job {
  char* host;
  const char* pin;
  size_t bytes, chunk, n, slots, parts;  // chunk = parts * kPart
  int helpers;                           // how many may join
  std::atomic<int> joined{0};
  std::atomic<size_t> next{0}, ready{0};  // parts taken, chunks landed
  std::atomic<size_t> done[kSlots];       // parts copied out of each slot
  bool exhausted() const { return next.load() >= n * parts; }
  // copies one part that has landed; false when there is none
  bool step()
  {
    size_t q = next.load();
    do {
      if (q >= ready.load(std::memory_order_acquire) * parts) return false;
    } while (!next.compare_exchange_weak(q, q + 1));
    const size_t ch = q / parts, o = (q % parts) * kPart, len = std::min(chunk, bytes - ch * chunk);
    if (o < len) std::memcpy(host + ch * chunk + o, pin + (ch % slots) * chunk + o, std::min(kPart, len - o));
    done[ch % slots].fetch_add(1, std::memory_order_release);
    return true;
  }
};

class Pool {
  std::mutex m;
  std::condition_variable cv;
  std::vector<Ring> idle;
  std::vector<std::shared_ptr<Job>> jobs;
  std::vector<std::thread> threads;
  int users = 0;
  int gen = 0;  // helpers of an earlier generation end

  void help(int mine)
  {
    std::unique_lock<std::mutex> l(m);
    for (;;) {
      std::shared_ptr<Job> j;
      cv.wait(l, [&]() {
        for (auto& c : jobs)
          if (!c->exhausted() && c->joined.load() < c->helpers) {
            j = c;
            return true;
          }
        return gen != mine;
      });
      if (!j) return;
      j->joined++;
      l.unlock();
      while (!j->exhausted())
        if (!j->step()) std::this_thread::yield();
      j.reset();
      l.lock();
    }
  }

public:
  Ring take(size_t bytes)
  {
    Ring r;
    {
      std::lock_guard<std::mutex> l(m);
      if (!idle.empty()) {
        r = idle.back();
        idle.pop_back();
      }
    }
    if (r.bytes >= bytes) return r;
    if (r.p) (void)hipHostFree(r.p);
    r = Ring{};
    if (hipHostMalloc((void**)&r.p, bytes, hipHostMallocPortable | hipHostMallocMapped) != hipSuccess) {
      (void)hipGetLastError();
      return Ring{};
    }
    if (hipHostGetDevicePointer((void**)&r.d, r.p, 0) != hipSuccess) {
      (void)hipGetLastError();
      (void)hipHostFree(r.p);
      return Ring{};
    }
    r.bytes = bytes;
    return r;
  }
  void give(Ring r)
  {
    {
      std::lock_guard<std::mutex> l(m);
      if (users > 0 && idle.size() < 2) {
        idle.push_back(r);
        return;
      }
    }
    (void)hipHostFree(r.p);
  }
  void add(const std::shared_ptr<Job>& j)
  {
    {
      std::lock_guard<std::mutex> l(m);
      const int most = std::min(j->helpers, (int)std::thread::hardware_concurrency() - 1);
      try {
        while ((int)threads.size() < most) threads.emplace_back([this, g = gen]() { help(g); });
      } catch (const std::system_error&) {  // fewer helpers, then
      }
      jobs.push_back(j);
    }
    cv.notify_all();
  }
  void remove(const std::shared_ptr<Job>& j)
  {
    std::lock_guard<std::mutex> l(m);
    jobs.erase(std::find(jobs.begin(), jobs.end(), j));
  }
  // a context begins (1) or ends (-1); the last one ends rings and threads
  void user(int d)
  {
    std::vector<Ring> rings;
    std::vector<std::thread> th;
    {
      std::lock_guard<std::mutex> l(m);
      users += d;
      if (users > 0) return;
      rings.swap(idle);
      th.swap(threads);
      gen++;
    }
    cv.notify_all();
    for (auto& t : th) t.join();
    for (auto& r : rings) (void)hipHostFree(r.p);
  }
};

inline Pool& pool()
{
  static Pool* p = new Pool;  // never destroyed: contexts may end in any order at exit
  return *p;
}

} // namespace dl
