// hostcopy.hpp -- copies between device memory and the caller's host arrays
// through pinned chunks.
//
// The caller's arrays are pageable and often fresh, so a plain copy is bound
// by one thread taking their page faults: 256 MiB into a new array took 27 ms
// (10 GB/s) with a 57 GB/s link, 1 MiB 0.63 ms.  Here the link fills pinned
// chunks and four threads move them on, so that the faults and the
// copies overlap with the link: 6.3-6.9 ms (39-42 GB/s), 64 MiB 7.4 -> 1.95
// ms, 9 MiB 0.89 -> 0.40 ms.  Chunks of 1 MiB reached 31 GB/s, of 2 and 4 MiB
// 39-42.  More than four threads gain 0 to 6%, and after eight the next
// solver's creation took 110 or, one time in three, 400 to 900 us.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <utility>

#include "errors.hpp"
#include "nflow.h"

namespace nflow {

// Runs f() on `extra` more threads (three at most) while this one runs
// mine(their number); fewer where threads or their memory cannot be had (f must
// do all the work that is left, whoever calls it).
template <class F, class Main>
void run_threads(int extra, F f, Main mine) {
  constexpr int MOST = 3;
  std::thread t[MOST];
  int n = 0;
  try {
    for (; n < std::min(extra, MOST); ++n) t[n] = std::thread(f);
  } catch (const std::exception&) {  // system_error or bad_alloc
  }
  mine(n);
  for (int i = 0; i < n; ++i) t[i].join();
}

// Helpers for a copy into the caller's pages; 0: too small for threads.  From
// 3 MiB they halve the time into fresh pages (8 MiB 1.9 -> 0.9 ms), and lose
// little where malloc hands the same pages out again (0.5 -> 0.7 ms).  1.7 MiB
// is 130 us as the runtime's own pageable copies, 310 us through the chunks.
inline int helpers_out(size_t bytes) {
  const unsigned hw = std::thread::hardware_concurrency();
  return bytes < (3u << 20) ? 0 : (int)std::min<size_t>(3, hw ? hw : 1);
}

// Helpers for a copy out of the caller's pages, which mostly are there: 67 MB
// 2.6 -> 1.95 ms, 323 MB 35 -> 8.2 (eight helpers: 1.98 and 8.3), but 9.5 MB 300
// us as the runtime's own copy and 370 to 750 through the chunks.
inline int helpers_in(size_t bytes) {
  const unsigned hw = std::thread::hardware_concurrency();
  return bytes < (32u << 20) ? 0 : (int)std::min<size_t>(3, hw ? hw : 1);
}

// memcpy by several threads (fresh destination pages are faulted in by all)
inline void parallel_memcpy(void* dst, const void* src, size_t n) {
  constexpr size_t PIECE = 1u << 20;
  std::atomic<size_t> next{0};
  auto work = [&] {
    for (size_t o; (o = next.fetch_add(PIECE)) < n;)
      std::memcpy(static_cast<char*>(dst) + o, static_cast<const char*>(src) + o, std::min(PIECE, n - o));
  };
  run_threads(helpers_out(n), work, [&](int) { work(); });
}

// Pinned host memory: a block for one short copy, or chunks and the events of
// the copies through them.
struct Pinned {
  static constexpr size_t CHUNK = 2u << 20, SLOTS = 8, BLOCK = 1u << 20;
  char* buf = nullptr;
  int device = -1;  // the events' device; -1: a block, without events
  hipEvent_t ev[SLOTS] = {};
  Pinned() = default;
  Pinned(const Pinned&) = delete;
  Pinned& operator=(const Pinned&) = delete;
  ~Pinned() {
    for (auto& e : ev)
      if (e) (void)hipEventDestroy(e);
    if (buf) (void)hipHostFree(buf);
  }
  bool open(int dev) {
    device = dev;
    bool ok = true;
    if (dev >= 0)
      for (auto& e : ev) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    void* p = nullptr;
    ok = ok && hipHostMalloc(&p, dev >= 0 ? SLOTS * CHUNK : BLOCK, hipHostMallocPortable) == hipSuccess;
    if (!ok) (void)hipGetLastError();
    buf = ok ? static_cast<char*>(p) : nullptr;
    return ok;
  }
};

// The process's pinned memory, at most 4 sets of chunks and 16 blocks (80 MiB),
// kept while any HostCopy lives and given back with the last: a new solver's
// first read-back finds it ready.  Copies that overlap each hold one of their
// own; those that find none left are plain ones.  (Sets made for a third copy
// at a time and freed after it: 8 threads that read 64^3 fields 1.9 ms at the
// 90th percentile, and 1.15 with plain copies alone.)
class PinnedPool {
 public:
  static std::shared_ptr<PinnedPool> get() {
    static std::mutex mu;
    static std::weak_ptr<PinnedPool> pool;
    std::lock_guard<std::mutex> lk(mu);
    std::shared_ptr<PinnedPool> p = pool.lock();
    if (!p) pool = p = std::make_shared<PinnedPool>();
    return p;
  }
  // a set of chunks for `device`
  std::unique_ptr<Pinned> take_chunks(int device) { return take(chunks_, device, true); }
  // a block; grow: make one where none is idle
  std::unique_ptr<Pinned> take_block(bool grow) { return take(blocks_, -1, grow); }
  void give(std::unique_ptr<Pinned> p) {
    std::lock_guard<std::mutex> lk(mu_);
    for (auto& q : p->device < 0 ? blocks_.idle : chunks_.idle)
      if (!q) {
        q = std::move(p);
        return;
      }
  }

 private:
  struct Kind {
    std::unique_ptr<Pinned> idle[16];
    int live, most;  // made and not freed; how many there may be
  };
  std::unique_ptr<Pinned> take(Kind& k, int device, bool grow) {
    std::unique_ptr<Pinned> other;  // another device's, in the way
    {
      std::lock_guard<std::mutex> lk(mu_);
      for (auto& p : k.idle)
        if (p && p->device == device) return std::move(p);
      if (!grow) return nullptr;
      if (k.live == k.most) {
        for (auto& p : k.idle)
          if (p && !other) other = std::move(p);
        if (!other) return nullptr;
        --k.live;
      }
      ++k.live;
    }
    other.reset();
    std::unique_ptr<Pinned> p(new (std::nothrow) Pinned);
    if (p && !p->open(device)) p.reset();
    if (!p) {
      std::lock_guard<std::mutex> lk(mu_);
      --k.live;
    }
    return p;
  }
  std::mutex mu_;
  Kind chunks_{{}, 0, 4}, blocks_{{}, 0, 16};
};

// One batch's copies: one host thread at a time, on the batch's stream and
// device.
class HostCopy {
 public:
  int device = 0;

  // `parts` consecutive ranges of n bytes from src on the device to dst[0],
  // dst[1], ...; complete on return, and so is all earlier work of the stream.
  int to_host(hipStream_t st, const void* src, size_t n, void* const* dst, int parts) {
    const size_t total = n * parts;
    const int helpers = helpers_out(total);
    const Lease lease(*this, helpers > 0 ? CHUNKS : total > Pinned::BLOCK ? NONE : total > TINY || !first_ ? GROW : IDLE);
    first_ = false;
    if (!lease) {  // plain copies
      for (int i = 0; i < parts; ++i)
        NFLOW_HIP(hipMemcpyAsync(dst[i], static_cast<const char*>(src) + i * n, n, hipMemcpyDeviceToHost, st));
      NFLOW_HIP(hipStreamSynchronize(st));
      return 0;
    }
    char* const buf = lease->buf;
    hipEvent_t* const ev = lease->ev;
    auto put = [&](size_t off, const char* from, size_t len) {  // [off, off + len) of the total
      while (len) {
        const size_t i = off / n, o = off % n, l = std::min(len, n - o);
        std::memcpy(static_cast<char*>(dst[i]) + o, from, l);
        off += l;
        from += l;
        len -= l;
      }
    };
    if (helpers == 0) {  // one short copy on the link (0.5 MiB: 69 us, as four plain ones 278 us)
      NFLOW_HIP(hipMemcpyAsync(buf, src, total, hipMemcpyDeviceToHost, st));
      NFLOW_HIP(hipStreamSynchronize(st));
      put(0, buf, total);
      return 0;
    }
    const size_t pieces = (total + PIECE - 1) / PIECE, chunks = (total + CHUNK - 1) / CHUNK;
    std::atomic<size_t> ready{0}, next{0};  // chunks on the host; next piece to move on
    std::atomic<size_t> moved[SLOTS];       // pieces moved out of each slot, over the whole copy
    for (auto& m : moved) m.store(0);
    std::atomic<bool> stop{false};
    auto move_on = [&](size_t i) {
      const size_t c = i / PER, off = i * PIECE;
      put(off, buf + (c % SLOTS) * CHUNK + (off - c * CHUNK), std::min(PIECE, total - off));
      moved[c % SLOTS].fetch_add(1, std::memory_order_release);
    };
    auto work = [&] {
      for (size_t i; !stop.load() && (i = next.fetch_add(1)) < pieces;) {
        while (ready.load(std::memory_order_acquire) <= i / PER) {
          if (stop.load()) return;
          std::this_thread::yield();
        }
        move_on(i);
      }
    };
    hipError_t err = hipSuccess;
    size_t issued = 0, done = 0;
    auto issue = [&] {  // keep half of the slots on the link, where they are free
      while (issued < chunks && issued < done + SLOTS / 2 && err == hipSuccess &&
             (issued < SLOTS || moved[issued % SLOTS].load(std::memory_order_acquire) >= (issued / SLOTS) * PER)) {
        const size_t off = issued * CHUNK;
        err = hipMemcpyAsync(buf + (issued % SLOTS) * CHUNK, static_cast<const char*>(src) + off,
                             std::min(CHUNK, total - off), hipMemcpyDeviceToHost, st);
        if (err == hipSuccess) err = hipEventRecord(ev[issued % SLOTS], st);
        ++issued;
      }
    };
    issue();
    run_threads(err == hipSuccess ? helpers : 0, work, [&](int running) {
      while (done < chunks && err == hipSuccess) {
        issue();
        if (err == hipSuccess && done < issued) {
          err = hipEventSynchronize(ev[done % SLOTS]);
          if (err != hipSuccess) break;
          ready.store(++done, std::memory_order_release);
          if (running == 0) {  // alone: move it on, with the next ones on the link
            issue();
            for (size_t i = next.load(); i < std::min(done * PER, pieces); ++i) {
              next.store(i + 1);
              move_on(i);
            }
          }
        } else if (err == hipSuccess) {
          std::this_thread::yield();
        }
      }
      if (err != hipSuccess)
        stop.store(true);
      else
        work();  // lend a hand with what is left
    });
    if (err != hipSuccess) {
      (void)hipStreamSynchronize(st);
      return fail(NFLOW_EDEVICE, "copy to the host: %s", hipGetErrorString(err));
    }
    return 0;
  }

  // n bytes from the host to dst on the device, in stream order; src is free
  // once the stream has been waited for.  (The chunks go back to the pool on
  // return, so a copy through them has ended then.)
  int to_device(hipStream_t st, void* dst, const void* src, size_t n) {
    const int most = helpers_in(n);
    const Lease lease(*this, most > 0 ? CHUNKS : NONE);
    if (!lease) {
      NFLOW_HIP(hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, st));
      return 0;
    }
    char* const buf = lease->buf;
    hipEvent_t* const ev = lease->ev;
    const size_t pieces = (n + PIECE - 1) / PIECE, chunks = (n + CHUNK - 1) / CHUNK;
    std::atomic<size_t> freed{0}, next{0};  // chunks that have left their slots; next piece to bring
    std::atomic<size_t> filled[SLOTS];      // pieces brought into each slot, over the whole copy
    for (auto& f : filled) f.store(0);
    std::atomic<bool> stop{false};
    auto bring = [&](size_t i) {
      const size_t c = i / PER, off = i * PIECE;
      std::memcpy(buf + (c % SLOTS) * CHUNK + (off - c * CHUNK), static_cast<const char*>(src) + off,
                  std::min(PIECE, n - off));
      filled[c % SLOTS].fetch_add(1, std::memory_order_release);
    };
    auto work = [&] {
      for (size_t i; !stop.load() && (i = next.fetch_add(1)) < pieces;) {
        while (i / PER >= freed.load(std::memory_order_acquire) + SLOTS) {
          if (stop.load()) return;
          std::this_thread::yield();
        }
        bring(i);
      }
    };
    hipError_t err = hipSuccess;
    run_threads(most, work, [&](int helpers) {
      for (size_t c = 0; c < chunks && err == hipSuccess; ++c) {
        // chunk c - SLOTS / 2 has left: its slot may be filled again
        if (c >= SLOTS / 2) {
          err = hipEventSynchronize(ev[(c - SLOTS / 2) % SLOTS]);
          if (err != hipSuccess) break;
          freed.store(c - SLOTS / 2 + 1, std::memory_order_release);
        }
        if (helpers == 0)
          for (size_t i; (i = next.load()) < std::min((c + 1) * PER, pieces);) {
            next.store(i + 1);
            bring(i);
          }
        const size_t mine = std::min<size_t>(PER, pieces - c * PER);
        while (filled[c % SLOTS].load(std::memory_order_acquire) < (c / SLOTS) * PER + mine) std::this_thread::yield();
        err = hipMemcpyAsync(static_cast<char*>(dst) + c * CHUNK, buf + (c % SLOTS) * CHUNK,
                             std::min(CHUNK, n - c * CHUNK), hipMemcpyHostToDevice, st);
        if (err == hipSuccess) err = hipEventRecord(ev[c % SLOTS], st);
      }
      if (err != hipSuccess) stop.store(true);
    });
    // the slots are free again only when the last chunks have left
    const hipError_t last = hipStreamSynchronize(st);
    if (err == hipSuccess) err = last;
    return err == hipSuccess ? 0 : fail(NFLOW_EDEVICE, "copy to the device: %s", hipGetErrorString(err));
  }

 private:
  static constexpr size_t CHUNK = Pinned::CHUNK, SLOTS = Pinned::SLOTS, PIECE = 256u << 10, PER = CHUNK / PIECE,
                          TINY = 4u << 10;
  std::shared_ptr<PinnedPool> pool_ = PinnedPool::get();
  // no copy to the host yet: a first one of up to TINY bytes that finds no idle
  // block goes plain (the first diagnostics of a process 190 -> 75 us; making a
  // block of 1 MiB takes some 70 us, a set of chunks 130)
  bool first_ = true;

  // what a copy takes from the pool: nothing, chunks, a block, a block only if one is idle
  enum Want { NONE, CHUNKS, GROW, IDLE };
  // a Pinned of the pool for one copy (where wanted and to be had); every copy
  // through it has ended when it goes back
  struct Lease {
    Lease(HostCopy& h, Want w)
        : pool(*h.pool_),
          p(w == NONE ? nullptr : w == CHUNKS ? pool.take_chunks(h.device) : pool.take_block(w == GROW)) {}
    ~Lease() {
      if (p) pool.give(std::move(p));
    }
    explicit operator bool() const { return p != nullptr; }
    Pinned* operator->() const { return p.get(); }
    PinnedPool& pool;
    std::unique_ptr<Pinned> p;
  };
};

}  // namespace nflow
