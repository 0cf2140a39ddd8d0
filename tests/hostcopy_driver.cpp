// csrc/hostcopy.hpp without a device (tests/test_hostcopy_cpu.py): run_threads
// when memory for a thread runs out (the threads that were started and the
// caller do the work, and nothing is thrown), and the pool's count of pinned
// memory over several devices, with the HIP calls it makes stood in for here.
#include <cstdio>
#include <cstdlib>
#include <new>

static long left = -1;  // allocations until one fails; < 0: none does
void* operator new(std::size_t n) {
  if (left >= 0 && left-- == 0) throw std::bad_alloc();
  return std::malloc(n);
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

#include "hostcopy.hpp"

static int pinned = 0, refuse = 0;
hipError_t hipHostMalloc(void** p, size_t, unsigned) {
  if (refuse) return hipErrorOutOfMemory;
  ++pinned;
  *p = std::malloc(1);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  --pinned;
  std::free(p);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(1);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }

static int pool() {
  using nflow::Pinned;
  using nflow::PinnedPool;
  {
    const auto p = PinnedPool::get();
    if (PinnedPool::get() != p) return 1;
    std::unique_ptr<Pinned> a[16];
    // one set for each of four devices, then a fifth device's in the place of one
    for (int d = 0; d < 4; ++d) a[d] = p->take_chunks(d);
    if (pinned != 4 || p->take_chunks(0)) return 2;
    for (int d = 0; d < 4; ++d) p->give(std::move(a[d]));
    a[0] = p->take_chunks(9);
    if (!a[0] || a[0]->device != 9 || pinned != 4) return 3;
    p->give(std::move(a[0]));
    // four of it in the end, and one that cannot be made is not counted
    for (int k = 0; k < 3; ++k) {
      refuse = k == 1;
      for (int i = 0; i < 4; ++i) a[i] = p->take_chunks(9);
      if (k != 1 && (!a[0] || !a[1] || !a[2] || !a[3] || p->take_chunks(9) || pinned != 4)) return 4;
      for (auto& x : a)
        if (x) p->give(std::move(x));
    }
    refuse = 0;
    if (p->take_block(false)) return 5;
    for (auto& x : a) x = p->take_block(true);
    if (pinned != 20 || p->take_block(true)) return 6;
    for (auto& x : a) p->give(std::move(x));
    if (!(a[0] = p->take_block(false)) || pinned != 20) return 7;
    p->give(std::move(a[0]));
  }
  return pinned == 0 ? 0 : 8;  // given back with the last holder
}

int main() {
  for (long k = 0; k < 4; ++k) {
    std::atomic<int> next{0}, done{0};
    auto work = [&] {
      while (next.fetch_add(1) < 1000) done.fetch_add(1);
    };
    int started = -1;
    left = k;
    nflow::run_threads(3, work, [&](int n) {
      left = -1;
      started = n;
      work();
    });
    if (done != 1000 || started != (k < 3 ? (int)k : 3)) return 1;
  }
  std::puts("threads ok");
  if (const int at = pool()) {
    std::printf("pool: check %d\n", at);
    return 1;
  }
  std::puts("pool ok");
  return 0;
}
