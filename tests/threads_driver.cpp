// run_threads (csrc/hostcopy.hpp) when memory for a thread runs out: the threads
// that were started and the caller do the work, and nothing is thrown
// (tests/test_hostcopy_cpu.py).
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
  return 0;
}
