// Copies between a caller's ordinary (pageable) host memory and the GPU.
//
// The runtime's own copy of pageable memory moves it through one thread and
// waits for each call.  Here chunks pass through a ring of pinned slots: the
// GPU fills (or drains) one slot while CPU threads copy others.  The threads
// of a large copy to the host first touch the pages of the result, which the
// caller's steps still queued on the GPU mostly hide: a fresh array's page
// faults cost as much as the copy.  Moments of 256^3 nodes, 268 MB: 26 ms ->
// 13 ms into a fresh array with nothing queued, 8 ms behind queued steps or
// into touched pages; of 256 x 128 x 128, 67 MB: 5.7 -> 2.5 ms; of 64^2: 62
// -> 27 us (one copy for both arrays).
//
// In between, where one thread would fault the pages of a fresh result in one
// by one, the runtime's copy stays, which pins them at once (2 MB into a
// fresh array 0.5 against 1.4 ms).
//
// Slots (one of 512 KiB for a small copy, a ring of 32 MiB for a large one)
// come from a pool; each call has its slots to itself, so calls of several
// threads and streams do not meet.  A ring costs 0.1 to 0.6 ms to pin and its
// first copy 1 to 5 ms more than the following ones, so
//  - the first is made once 4 small copies or 64 MiB have gone by, before
//    which the runtime copies;
//  - at most 8 and 2 of them exist (68 MiB): a call that finds none free
//    leaves its copy to the runtime;
//  - when the last context goes, one of each kind stays if a copy asked for it
//    since the last time, and goes too if none did.
// So a program that makes a lattice, reads it and destroys it, again and again,
// finds its slots there.  Its read-back, by the runtime / through slots made
// anew for each / so: 9 MiB 0.58 / 1.7 / 0.57 ms, 33 MiB 2.0 / 6.4 / 1.0, 256
// MiB 26 / 25 / 12.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "lbm_internal.h"

namespace lbm {
namespace {

constexpr int kSlots = 8;
// below this the runtime's copy is as fast (64 KiB: 12 us either way)
constexpr size_t kDirect = 64u << 10;
// from here on several threads pay for their start (about 0.1 ms)
constexpr size_t kThreaded = 8u << 20;
constexpr int kWorkers = 6;
// a small copy takes one slot, a large one chunks of an eighth of it, up to
// what a slot holds, so that little goes to the chunks' events (268 MB in
// chunks of 1 MiB: 10.5 ms, of 4 MiB: 8.9)
constexpr size_t kSmallSlot = 512u << 10, kLargeSlot = 4u << 20;
inline size_t chunk_bytes(size_t bytes) {
  return std::min((bytes / kSlots + 4095) / 4096 * 4096, kLargeSlot);
}
// the runtime's upload of pageable memory is as fast up to here (9.4 MB: 355
// against 485 us, 36 MB: 1350 / 1150, 318 MB: 19.4 / 12 ms)
constexpr size_t kFeed = 32u << 20;

struct Slots {
  int device;
  bool large;
  char* base;
  hipEvent_t ev[kSlots];
};

void free_slots(const Slots& r) {
  for (hipEvent_t e : r.ev)
    if (e) (void)hipEventDestroy(e);
  if (r.base) (void)hipHostFree(r.base);
}

// The slots of one kind, in use and idle.
struct Pool {
  const int most;     // so many at a time
  const size_t earn;  // copies (small) or bytes (large) until the first is made
  int made = 0;
  size_t went = 0;    // copies or bytes so far
  bool used = false;  // a copy came since the last context went
  std::vector<Slots> idle;
};
constexpr int kMostSmall = 8, kMostLarge = 2;
std::mutex g_pool_mutex;
Pool g_small{kMostSmall, 4, 0, 0, false, {}};
Pool g_large{kMostLarge, 64u << 20, 0, 0, false, {}};
int64_t g_contexts = 0;

// Slots (with an event each for a large copy) for one call, or none: then
// the runtime copies.
struct Ring {
  Slots r{};
  bool ok = false;
  Ring(bool large, size_t bytes) {
    Pool& pool = large ? g_large : g_small;
    r.large = large;
    if (hipGetDevice(&r.device) != hipSuccess) return;
    {
      std::lock_guard<std::mutex> lk(g_pool_mutex);
      pool.went += large ? bytes : 1;
      pool.used = true;
      for (size_t k = 0; k < pool.idle.size(); ++k)
        if (pool.idle[k].device == r.device) {
          r = pool.idle[k];
          pool.idle.erase(pool.idle.begin() + (std::ptrdiff_t)k);
          ok = true;
          return;
        }
      if (pool.made >= pool.most || pool.went < pool.earn) return;
      pool.idle.reserve((size_t)pool.most);  // giving back allocates nothing
      ++pool.made;
    }
    ok = hipHostMalloc((void**)&r.base, large ? kSlots * kLargeSlot : kSmallSlot,
                       hipHostMallocDefault) == hipSuccess;
    if (!ok) r.base = nullptr;
    for (hipEvent_t& e : r.ev)
      if (ok && large) ok = hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (!ok) (void)hipGetLastError();
    std::lock_guard<std::mutex> lk(g_pool_mutex);
    if (!ok) {
      --pool.made;
      pool.went = 0;
      free_slots(r);
    }
  }
  Ring(const Ring&) = delete;
  Ring& operator=(const Ring&) = delete;
  ~Ring() {
    if (!ok) return;
    std::lock_guard<std::mutex> lk(g_pool_mutex);
    (r.large ? g_large : g_small).idle.push_back(r);
  }
  char* slot(size_t j) const { return r.base + (j % kSlots) * kLargeSlot; }
  hipEvent_t event(size_t j) const { return r.ev[j % kSlots]; }
};

// What the threads of a copy wait for: chunks below `open` may be taken.
// The first of them comes behind everything that the stream still has to do,
// so a thread sleeps until then; afterwards its next chunk is a few DMAs of
// 0.1 ms away, and a thread looks for that long before it sleeps (64 MiB 2.9
// ms where it slept at once, 2.4 so).  Threads that only yielded kept six
// CPUs busy for as long as the steps before a result took.
class Gate {
 public:
  explicit Gate(size_t open) : open_(open) {}
  // chunks below n are there
  void raise(size_t n) {
    {
      std::lock_guard<std::mutex> lk(m_);
      open_.store(n, std::memory_order_release);
    }
    cv_.notify_all();
  }
  void stop() {
    {
      std::lock_guard<std::mutex> lk(m_);
      stop_.store(true, std::memory_order_release);
    }
    cv_.notify_all();
  }
  bool stopped() const { return stop_.load(std::memory_order_acquire); }
  // Returns when chunk j is there (true) or the copy is given up.
  bool wait(size_t j) {
    if (open_.load(std::memory_order_acquire) > 0) {
      const auto until = std::chrono::steady_clock::now() + kLook;
      do {
        if (open_.load(std::memory_order_acquire) > j) return true;
        if (stopped()) return false;
        std::this_thread::yield();
      } while (std::chrono::steady_clock::now() < until);
    }
    std::unique_lock<std::mutex> lk(m_);
    cv_.wait(lk, [&] { return stopped() || open_.load(std::memory_order_relaxed) > j; });
    return open_.load(std::memory_order_relaxed) > j;
  }

 private:
  static constexpr std::chrono::microseconds kLook{1000};
  std::mutex m_;
  std::condition_variable cv_;
  std::atomic<size_t> open_;
  std::atomic<bool> stop_{false};
};

// Threads that run fn until the object goes; none where they cannot start.
struct Crew {
  std::vector<std::thread> t;
  Gate& gate;
  template <class Fn>
  Crew(Gate& g, int n, Fn fn) : gate(g) {
    t.reserve((size_t)n);
    for (int k = 0; k < n; ++k) {
      try {
        t.emplace_back(fn);
      } catch (...) {
        break;
      }
    }
  }
  ~Crew() {
    gate.stop();
    for (std::thread& x : t) x.join();
  }
};

// Bytes [a, b) of the pieces laid end to end, to or from `chunk`.
void move_pieces(const HostPiece* pieces, int count, size_t a, size_t b, char* chunk, bool out) {
  size_t at = 0;
  for (int k = 0; k < count; ++k) {
    const size_t lo = std::max(a, at), hi = std::min(b, at + pieces[k].bytes);
    if (lo < hi) {
      char* host = (char*)pieces[k].p + (lo - at);
      if (out)
        std::memcpy(host, chunk + (lo - a), hi - lo);
      else
        std::memcpy(chunk + (lo - a), host, hi - lo);
    }
    at += pieces[k].bytes;
  }
}

int plain(char* dev, const HostPiece* pieces, int count, bool out, hipStream_t s) {
  for (int k = 0; k < count; ++k) {
    if (pieces[k].bytes)
      LBM_HIP(out ? hipMemcpyAsync(pieces[k].p, dev, pieces[k].bytes, hipMemcpyDeviceToHost, s)
                  : hipMemcpyAsync(dev, pieces[k].p, pieces[k].bytes, hipMemcpyHostToDevice, s));
    dev += pieces[k].bytes;
  }
  LBM_HIP(hipStreamSynchronize(s));
  return LBM_OK;
}

void pause() { std::this_thread::yield(); }

// Ordinary memory, which the slots are for.  What the caller allocated
// pinned, managed or on the GPU the runtime copies directly (256 MiB into
// pinned memory 4.9 ms, through the slots 9.4), and CPU threads need not be
// able to reach it.  0.4 us a question.
bool ordinary(const HostPiece* pieces, int count) {
  for (int k = 0; k < count; ++k) {
    if (!pieces[k].bytes) continue;
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, pieces[k].p) != hipSuccess)
      (void)hipGetLastError();
    else if (a.type != hipMemoryTypeUnregistered)
      return false;
  }
  return true;
}

// Touches the pages of the pieces without changing what they hold, block by
// block by the threads that draw them; returns when all blocks are done (a
// copy into pages that another thread still touches would lose bytes) or
// stop is set.
struct Toucher {
  static constexpr size_t kBlock = 2u << 20, kPage = 4096;
  const HostPiece* pieces;
  int count;
  size_t blocks = 0;
  std::atomic<size_t> next{0}, done{0};
  Toucher(const HostPiece* p, int n) : pieces(p), count(n) {
    for (int k = 0; k < n; ++k) blocks += (p[k].bytes + kBlock - 1) / kBlock;
  }
  void block(size_t j) {
    for (int k = 0; k < count; ++k) {
      const size_t here = (pieces[k].bytes + kBlock - 1) / kBlock;
      if (j >= here) {
        j -= here;
        continue;
      }
      char* p = (char*)pieces[k].p;
      const size_t end = std::min(pieces[k].bytes, (j + 1) * kBlock);
      for (size_t i = j * kBlock; i < end; i += kPage) {
        volatile char* q = p + i;
        *q = *q;  // a store, which volatile keeps
      }
      return;
    }
  }
  void run(const Gate& gate) {
    for (size_t j; (j = next.fetch_add(1)) < blocks;) {
      if (!gate.stopped()) block(j);
      done.fetch_add(1, std::memory_order_release);
    }
    while (done.load(std::memory_order_acquire) < blocks && !gate.stopped()) pause();
  }
};

// GPU -> host: slot after slot is filled in stream order; the crew (or this
// thread) empties those that are there.
int drain(const char* dev, const HostPiece* pieces, int count, size_t bytes, const Ring& r,
          hipStream_t s) {
  if (!r.r.large) {
    LBM_HIP(hipMemcpyAsync(r.slot(0), dev, bytes, hipMemcpyDeviceToHost, s));
    LBM_HIP(hipStreamSynchronize(s));
    move_pieces(pieces, count, 0, bytes, r.slot(0), true);
    return LBM_OK;
  }
  const size_t chunk = chunk_bytes(bytes), n = (bytes + chunk - 1) / chunk;
  auto end = [&](size_t j) { return std::min(bytes, (j + 1) * chunk); };
  auto issue = [&](size_t j) -> hipError_t {
    const hipError_t e = hipMemcpyAsync(r.slot(j), dev + j * chunk, end(j) - j * chunk,
                                        hipMemcpyDeviceToHost, s);
    return e == hipSuccess ? hipEventRecord(r.event(j), s) : e;
  };
  std::vector<std::atomic<bool>> out(n);  // copied out of its slot
  std::atomic<size_t> next{0};
  Gate arrived(0);
  Toucher toucher(pieces, count);
  auto copy = [&](size_t j) {
    move_pieces(pieces, count, j * chunk, end(j), r.slot(j), true);
    out[j].store(true, std::memory_order_release);
  };
  auto work = [&]() {
    toucher.run(arrived);
    for (size_t j; (j = next.fetch_add(1)) < n && arrived.wait(j);) copy(j);
  };
  Crew crew(arrived, kWorkers, work);
  for (size_t j = 0; j < n && j < kSlots; ++j) LBM_HIP(issue(j));
  for (size_t j = 0; j < n; ++j) {
    LBM_HIP(hipEventSynchronize(r.event(j)));
    arrived.raise(j + 1);
    if (crew.t.empty()) copy(j);
    // the slot takes chunk j + kSlots once its own is out; the crew is
    // several chunks behind at most, so look at the oldest first
    if (j + kSlots < n) {
      while (!out[j].load(std::memory_order_acquire)) pause();
      LBM_HIP(issue(j + kSlots));
    }
  }
  for (size_t j = n > kSlots ? n - kSlots : 0; j < n; ++j)
    while (!out[j].load(std::memory_order_acquire)) pause();
  return LBM_OK;
}

// Host -> GPU, the other way round.
int feed(char* dev, const HostPiece* pieces, int count, size_t bytes, const Ring& r,
         hipStream_t s) {
  const size_t chunk = chunk_bytes(bytes), n = (bytes + chunk - 1) / chunk;
  auto end = [&](size_t j) { return std::min(bytes, (j + 1) * chunk); };
  std::vector<std::atomic<bool>> full(n);
  std::atomic<size_t> next{0};
  Gate free(std::min<size_t>(n, kSlots));
  auto fill = [&](size_t j) {
    move_pieces(pieces, count, j * chunk, end(j), r.slot(j), false);
    full[j].store(true, std::memory_order_release);
  };
  auto work = [&]() {
    for (size_t j; (j = next.fetch_add(1)) < n && free.wait(j);) fill(j);
  };
  Crew crew(free, kWorkers, work);
  for (size_t j = 0; j < n; ++j) {
    if (j >= kSlots) {
      LBM_HIP(hipEventSynchronize(r.event(j)));
      free.raise(j + 1);
    }
    if (crew.t.empty()) fill(j);
    while (!full[j].load(std::memory_order_acquire)) pause();
    LBM_HIP(hipMemcpyAsync(dev + j * chunk, r.slot(j), end(j) - j * chunk, hipMemcpyHostToDevice, s));
    LBM_HIP(hipEventRecord(r.event(j), s));
  }
  LBM_HIP(hipStreamSynchronize(s));
  return LBM_OK;
}

int transfer(char* dev, const HostPiece* pieces, int count, bool out, hipStream_t s) {
  size_t bytes = 0;
  for (int k = 0; k < count; ++k) bytes += pieces[k].bytes;
  const bool large = bytes >= (out ? kThreaded : kFeed);
  const bool small = out && bytes >= kDirect && bytes <= kSmallSlot;
  if ((!large && !small) || !ordinary(pieces, count)) return plain(dev, pieces, count, out, s);
  Ring ring(large, bytes);
  if (!ring.ok) return plain(dev, pieces, count, out, s);
  const int rc = out ? drain(dev, pieces, count, bytes, ring, s)
                     : feed(dev, pieces, count, bytes, ring, s);
  // after a failure nothing may still move through the slots
  if (rc) (void)hipStreamSynchronize(s);
  return rc;
}

}  // namespace

int copy_to_host(const void* dev, const HostPiece* pieces, int count, hipStream_t s) {
  return transfer((char*)const_cast<void*>(dev), pieces, count, true, s);
}

int copy_to_device(void* dev, const void* host, size_t bytes, hipStream_t s) {
  const HostPiece p{const_cast<void*>(host), bytes};
  return transfer((char*)dev, &p, 1, false, s);
}

int copy_to_host_plain(const void* dev, const HostPiece* pieces, int count, hipStream_t s) {
  return plain((char*)const_cast<void*>(dev), pieces, count, true, s);
}

void transfer_context(int delta) {
  Slots drop[kMostSmall + kMostLarge];
  size_t count = 0;
  {
    std::lock_guard<std::mutex> lk(g_pool_mutex);
    g_contexts += delta;
    if (g_contexts > 0 || delta > 0) return;
    for (Pool* pool : {&g_small, &g_large}) {
      const size_t keep = pool->used ? 1 : 0;
      while (pool->idle.size() > keep) {
        drop[count++] = pool->idle.back();
        pool->idle.pop_back();
        --pool->made;
      }
      if (!pool->used) pool->went = 0;
      pool->used = false;
    }
  }
  for (size_t k = 0; k < count; ++k) free_slots(drop[k]);
}

}  // namespace lbm
