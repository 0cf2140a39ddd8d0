// hostcopy.hpp -- copies between device memory and the caller's host arrays
// through pinned chunks.
//
// The caller's arrays are pageable and often fresh, so a plain copy is bound
// by one thread taking their page faults: 256 MiB into a new array took 27 ms
// (10 GB/s) with a 57 GB/s link, 1 MiB 0.63 ms.  Here the link fills pinned
// chunks and up to eight threads move them on, so that the faults and the
// copies overlap with the link: 6.3-6.9 ms (39-42 GB/s), 64 MiB 7.4 -> 1.95
// ms, 9 MiB 0.89 -> 0.40 ms.  Chunks of 1 MiB reached 31 GB/s, of 2 and 4 MiB
// 39-42; four threads are as good as twelve for 256 MiB, eight best at 9 MiB.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <memory>
#include <new>
#include <system_error>
#include <thread>

#include "errors.hpp"
#include "nflow.h"

namespace nflow {

// Runs f() on `extra` more threads and on this one; fewer where threads
// cannot be had (f must do all the work that is left, whoever calls it).
template <class F, class Main>
void run_threads(int extra, F f, Main mine) {
  constexpr int MOST = 8;
  std::thread t[MOST];
  int n = 0;
  try {
    for (; n < std::min(extra, MOST); ++n) t[n] = std::thread(f);
  } catch (const std::system_error&) {
  }
  mine(n);
  for (int i = 0; i < n; ++i) t[i].join();
}

inline int copy_threads(size_t bytes) {
  const unsigned hw = std::thread::hardware_concurrency();
  return (int)std::min<size_t>({bytes >> 20, 8, hw ? hw : 1});
}

// memcpy by several threads (fresh destination pages are faulted in by all)
inline void parallel_memcpy(void* dst, const void* src, size_t n) {
  constexpr size_t PIECE = 1u << 20;
  std::atomic<size_t> next{0};
  auto work = [&] {
    for (size_t o; (o = next.fetch_add(PIECE)) < n;)
      std::memcpy(static_cast<char*>(dst) + o, static_cast<const char*>(src) + o, std::min(PIECE, n - o));
  };
  run_threads(copy_threads(n) - 1, work, [&](int) { work(); });
}

// The pinned chunks of one batch: used by one host thread at a time, on the
// batch's stream.  16 MiB, taken at the first copy and held as the export
// scratch on the device is.
class HostCopy {
 public:
  HostCopy() = default;
  HostCopy(const HostCopy&) = delete;
  HostCopy& operator=(const HostCopy&) = delete;
  ~HostCopy() {
    for (auto& e : ev_)
      if (e) (void)hipEventDestroy(e);
    if (buf_) (void)hipHostFree(buf_);
  }

  // `parts` consecutive ranges of n bytes from src on the device to dst[0],
  // dst[1], ...; complete on return, and so is all earlier work of the stream.
  int to_host(hipStream_t st, const void* src, size_t n, void* const* dst, int parts) {
    const size_t total = n * parts;
    if (!open()) {  // no pinned memory: plain copies
      for (int i = 0; i < parts; ++i)
        NFLOW_HIP(hipMemcpyAsync(dst[i], static_cast<const char*>(src) + i * n, n, hipMemcpyDeviceToHost, st));
      NFLOW_HIP(hipStreamSynchronize(st));
      return 0;
    }
    auto put = [&](size_t off, const char* from, size_t len) {  // [off, off + len) of the total
      while (len) {
        const size_t i = off / n, o = off % n, l = std::min(len, n - o);
        std::memcpy(static_cast<char*>(dst[i]) + o, from, l);
        off += l;
        from += l;
        len -= l;
      }
    };
    if (total <= PIECE) {
      NFLOW_HIP(hipMemcpyAsync(buf_, src, total, hipMemcpyDeviceToHost, st));
      NFLOW_HIP(hipStreamSynchronize(st));
      put(0, buf_, total);
      return 0;
    }
    const size_t pieces = (total + PIECE - 1) / PIECE;
    std::atomic<size_t> ready{0}, next{0};  // chunks on the host; next piece to move on
    std::atomic<size_t> moved[SLOTS];       // pieces moved out of each slot, over the whole copy
    for (auto& m : moved) m.store(0);
    std::atomic<bool> stop{false};
    auto work = [&] {
      for (size_t i; !stop.load() && (i = next.fetch_add(1)) < pieces;) {
        const size_t c = i / PER, off = i * PIECE;
        while (ready.load(std::memory_order_acquire) <= c) {
          if (stop.load()) return;
          std::this_thread::yield();
        }
        put(off, buf_ + (c % SLOTS) * CHUNK + (off - c * CHUNK), std::min(PIECE, total - off));
        moved[c % SLOTS].fetch_add(1, std::memory_order_release);
      }
    };
    hipError_t err = hipSuccess;
    run_threads(copy_threads(total), work, [&](int helpers) {
      const size_t chunks = (total + CHUNK - 1) / CHUNK;
      size_t issued = 0, done = 0;
      auto slot_free = [&](size_t c) {  // every earlier chunk of the slot moved on?
        return c < SLOTS || moved[c % SLOTS].load(std::memory_order_acquire) >= (c / SLOTS) * PER;
      };
      while (done < chunks && err == hipSuccess) {
        while (issued < chunks && issued < done + SLOTS / 2 && slot_free(issued) && err == hipSuccess) {
          const size_t off = issued * CHUNK;
          err = hipMemcpyAsync(buf_ + (issued % SLOTS) * CHUNK, static_cast<const char*>(src) + off,
                               std::min(CHUNK, total - off), hipMemcpyDeviceToHost, st);
          if (err == hipSuccess) err = hipEventRecord(ev_[issued % SLOTS], st);
          ++issued;
        }
        if (err == hipSuccess && done < issued) {
          err = hipEventSynchronize(ev_[done % SLOTS]);
          if (err == hipSuccess) ready.store(++done, std::memory_order_release);
          if (helpers == 0 && err == hipSuccess)  // alone: move it on before the next
            for (size_t i; (i = next.load()) < std::min(done * PER, pieces);) {
              next.store(i + 1);
              const size_t c = i / PER, off = i * PIECE;
              put(off, buf_ + (c % SLOTS) * CHUNK + (off - c * CHUNK), std::min(PIECE, total - off));
              moved[c % SLOTS].fetch_add(1, std::memory_order_release);
            }
        } else if (err == hipSuccess) {
          std::this_thread::yield();
        }
      }
      if (err != hipSuccess) stop.store(true);
      else work();  // lend a hand with what is left
    });
    if (err != hipSuccess) {
      (void)hipStreamSynchronize(st);
      return fail(NFLOW_EDEVICE, "copy to the host: %s", hipGetErrorString(err));
    }
    return 0;
  }

  // n bytes from the host to dst on the device, in stream order; src may be
  // reused on return (the last chunks may still be on their way).
  int to_device(hipStream_t st, void* dst, const void* src, size_t n) {
    if (n <= CHUNK || !open()) {
      NFLOW_HIP(hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, st));
      NFLOW_HIP(hipStreamSynchronize(st));
      return 0;
    }
    const size_t pieces = (n + PIECE - 1) / PIECE, chunks = (n + CHUNK - 1) / CHUNK;
    std::atomic<size_t> freed{0}, next{0};  // chunks that have left their slots; next piece to bring
    std::atomic<size_t> filled[SLOTS];      // pieces brought into each slot, over the whole copy
    for (auto& f : filled) f.store(0);
    std::atomic<bool> stop{false};
    auto bring = [&](size_t i) {
      const size_t c = i / PER, off = i * PIECE;
      std::memcpy(buf_ + (c % SLOTS) * CHUNK + (off - c * CHUNK), static_cast<const char*>(src) + off,
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
    run_threads(copy_threads(n), work, [&](int helpers) {
      for (size_t c = 0; c < chunks && err == hipSuccess; ++c) {
        // chunk c - SLOTS / 2 has left: its slot may be filled again
        if (c >= SLOTS / 2) {
          err = hipEventSynchronize(ev_[(c - SLOTS / 2) % SLOTS]);
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
        err = hipMemcpyAsync(static_cast<char*>(dst) + c * CHUNK, buf_ + (c % SLOTS) * CHUNK,
                             std::min(CHUNK, n - c * CHUNK), hipMemcpyHostToDevice, st);
        if (err == hipSuccess) err = hipEventRecord(ev_[c % SLOTS], st);
      }
      if (err != hipSuccess) stop.store(true);
    });
    // the slots are free again only when the last chunks have left
    const hipError_t last = hipStreamSynchronize(st);
    if (err == hipSuccess) err = last;
    return err == hipSuccess ? 0 : fail(NFLOW_EDEVICE, "copy to the device: %s", hipGetErrorString(err));
  }

 private:
  static constexpr size_t CHUNK = 2u << 20, SLOTS = 8, PIECE = 256u << 10, PER = CHUNK / PIECE;
  char* buf_ = nullptr;
  hipEvent_t ev_[SLOTS] = {};
  bool failed_ = false;

  bool open() {
    if (buf_) return true;
    if (failed_) return false;
    bool ok = true;
    for (auto& e : ev_) ok = ok && (e || hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess);
    void* p = nullptr;
    ok = ok && hipHostMalloc(&p, SLOTS * CHUNK, hipHostMallocPortable) == hipSuccess;
    if (!ok) {
      (void)hipGetLastError();
      failed_ = true;
      return false;
    }
    buf_ = static_cast<char*>(p);
    return true;
  }
};

}  // namespace nflow
