// The plan of two-step launches (csrc/sweep_plan.cpp) for a batch given as
// arguments (tests/test_sweep_plan_cpu.py): CUs, nflow_tuning.temporal, then
// nx ny nz casetype per lattice.  Prints "tx tz h workgroups" per lattice (one
// line "none" without a plan, "small" and the nodes of the largest where the
// lattices run in k_small) after checking the work list: tiles within the
// kernel's limits, each node in exactly one.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "sweep_plan.hpp"

#define CHECK(c)                                                         \
  do {                                                                   \
    if (!(c)) {                                                          \
      std::fprintf(stderr, "check failed at line %d: %s\n", __LINE__, #c); \
      std::exit(1);                                                      \
    }                                                                    \
  } while (0)

int main(int argc, char** argv) {
  using namespace nflow;
  std::vector<nflow_input> in;
  for (int a = 3; a + 3 < argc; a += 4) {
    nflow_input i{};
    i.nx = std::atoi(argv[a]);
    i.ny = std::atoi(argv[a + 1]);
    i.nz = std::atoi(argv[a + 2]);
    i.casetype = std::atoi(argv[a + 3]);
    in.push_back(i);
  }
  if (const int n = small_plan(in, std::atoi(argv[1]), std::atoi(argv[2]))) {
    std::printf("small %d\n", n);
    return 0;
  }
  const auto plan = sweep_plan(in, std::atoi(argv[1]), std::atoi(argv[2]));
  if (plan.empty()) {
    std::puts("none");
    return 0;
  }
  const auto work = sweep_work(in, plan);
  CHECK(plan.size() == in.size() && work.size() % 8 == 0);
  for (size_t i = 0; i < in.size(); ++i) {
    const nflow_input& l = in[i];
    const SweepShape& s = plan[i];
    std::vector<unsigned char> seen((size_t)((l.nx - 1) / s.tx + 1) * ((l.nz - 1) / s.tz + 1) * ((l.ny - 1) / s.h + 1));
    long wgs = 0;
    for (const SweepItem& w : work) {
      if (w.h == 0 || w.lat != (int)i) continue;
      ++wgs;
      CHECK(w.tx == s.tx && w.tz == s.tz && w.h == s.h);
      CHECK(w.tx * w.tz <= SWEEP_NT && w.tz <= SWEEP_ROWS);
      CHECK(w.tz * (w.tx + 2) <= SWEEP_SLOT0 && (w.tz + 1) * (w.tx + 2) <= SWEEP_SLOT1);
      CHECK(2 * (w.tx + 2) + 2 * w.tz <= SWEEP_NT);  // one halo node per thread
      // its farthest byte: the last node of planes ya - 2 .. ya + h + 1 in blocks
      // of 19 runs of 64 nodes, from the block that the first one lies in
      const long long nxz = (long long)l.nx * l.nz, from = std::max(w.ya - 2, 0) * nxz / 64 * 64;
      const long long n = std::min<long long>(l.ny, (long long)w.ya + w.h + 2) * nxz - 1 - from;
      CHECK(((n / 64 * 19 + 18) * 64 + n % 64) * 4 + 3 < 1ll << 32);
      CHECK(w.x0 % s.tx == 0 && w.z0 % s.tz == 0 && w.ya % s.h == 0 && w.x0 < l.nx && w.z0 < l.nz && w.ya < l.ny);
      unsigned char& at = seen[(size_t)(w.x0 / s.tx) + (size_t)((l.nx - 1) / s.tx + 1) *
                                   ((size_t)(w.z0 / s.tz) + (size_t)((l.nz - 1) / s.tz + 1) * (w.ya / s.h))];
      CHECK(!at);
      at = 1;
    }
    CHECK(wgs == s.wgs && wgs == (long)seen.size());
    std::printf("%d %d %d %ld\n", s.tx, s.tz, s.h, s.wgs);
  }
  return 0;
}
