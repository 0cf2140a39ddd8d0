// sweep_plan.cpp -- tiles and chunk heights of two-step launches (k_sweep), and
// where they pay.
#include "sweep_plan.hpp"

#include <algorithm>
#include <cstddef>
#include <utility>

namespace nflow {

// A workgroup of k_sweep reads planes ya - 2 .. ya + h + 1 through a window of
// 32-bit byte offsets that starts at the first plane's block of 64 nodes: its
// farthest element is run 18 of node (h + 4) nxz + 62 of the window, 19 (h + 4)
// nxz + 19 x 62 + 18 x 64 at most.
int sweep_max_height(const nflow_input& in) {
  constexpr long long nodes = ((1ll << 30) - 1 - 19 * 62 - 18 * 64) / 19;
  return (int)std::max(0ll, nodes / ((long long)in.nx * in.nz) - 4);
}

// Chunks of at most h planes, evened out over y.
static int even_height(int ny, int h) {
  const int nch = (ny - 1) / h + 1;
  return (ny - 1) / nch + 1;
}

// One workgroup fills a CU (its LDS).  It sweeps its h planes, plus 0.28 for
// the planes around the chunk that it only takes the first step on, at
//   3.58 + 0.22 halo + w (3.06 fill m + x) us a plane
// (x 1.05 for channels), halo and fill the halo and own nodes per thread, m =
// 1.32 where rows do not start on 128-byte lines, x = 0.97 for tiles split in
// x, 2.04 where the splits are off 64-byte boundaries, and 3.1 us for its
// start.  Fitted, with 4 us a launch and 6% for more than one round of
// workgroups, to 600 launches of 62 cavities and channels of 40^3 to 512^3
// nodes at up to 18 shapes each (9% rms); the shape it picks is within 1.2% of
// the fastest measured one on average, and within 12%.
static SweepShape sweep_shape(const nflow_input& in, int tx, int tz, int h) {
  SweepShape s;
  const int ntx = (in.nx + tx - 1) / tx, ntz = (in.nz + tz - 1) / tz, nch = (in.ny - 1) / h + 1;
  s.tx = tx;
  s.tz = tz;
  s.h = h;
  s.wgs = (long)ntx * ntz * nch;
  const double halo = ((ntz > 1 ? 2.0 * (tx + 2) : 0.0) + (ntx > 1 ? 2.0 * tz : 0.0)) / SWEEP_NT;
  const double fill = (double)tx * tz / SWEEP_NT, split = ntx == 1 ? 0.0 : tx % 16 ? 2.04 : 0.97;
  const double planes = ((double)in.ny / nch + 0.28) * (in.casetype == NFLOW_CHANNEL ? 1.05 : 1.0);
  s.us0 = 3.1 + planes * (3.58 + 0.22 * halo);
  s.us1 = planes * (3.06 * fill * (in.nx % 32 ? 1.32 : 1.0) + split);
  return s;
}
static constexpr double SWEEP_LAUNCH_US = 4.0, SWEEP_ROUNDS = 1.06;

// us of one step per launch of one lattice, and 3 us a launch: 39 nodes per
// ns, 12% less where rows do not start on 128-byte lines
static double one_step_us(const nflow_input& in) {
  return (double)in.nx * in.ny * in.nz / 39.0e3 * (in.nx % 32 ? 1.12 : 1.0);
}
static constexpr double ONE_STEP_LAUNCH_US = 3.0;

// The candidate tile shapes of a lattice: whole x rows where three of them
// fit the exchange, and widths of 64-byte multiples; as many rows as fit,
// evened out over z.
static std::vector<std::pair<int, int>> sweep_tiles(const nflow_input& in) {
  std::vector<std::pair<int, int>> out;
  auto add = [&](int tx) {
    const int tz = std::min({in.nz, (int)SWEEP_ROWS, SWEEP_NT / tx, SWEEP_SLOT0 / (tx + 2), SWEEP_SLOT1 / (tx + 2) - 1});
    const int ntz = (in.nz + tz - 1) / tz;
    out.emplace_back(tx, (in.nz + ntz - 1) / ntz);
  };
  constexpr int WIDEST = SWEEP_SLOT1 / 4 - 2;  // three rows
  if (in.nx <= WIDEST) add(in.nx);
  for (int tx = 80; tx <= WIDEST && tx < in.nx; tx += 16) add(tx);
  return out;
}

std::vector<SweepShape> sweep_plan(const std::vector<nflow_input>& lats, int cu_count, int temporal) {
  std::vector<SweepShape> none;
  // a chunk height is a choice for one lattice; batches of several choose
  // for themselves or not at all
  if (temporal == 0 || lats.empty() || (temporal > 0 && lats.size() != 1)) return none;
  for (const auto& in : lats)
    if (in.casetype == NFLOW_PIPE || sweep_max_height(in) < std::max(temporal, 1)) return none;
  std::vector<SweepShape> shape(lats.size());
  double single = 2.0 * ONE_STEP_LAUNCH_US, pair = SWEEP_LAUNCH_US;  // us of two steps, either way
  if (lats.size() == 1) {
    const nflow_input& in = lats[0];
    double best = 1e30;
    for (const auto& tile : sweep_tiles(in)) {
      const long cols = (long)((in.nx + tile.first - 1) / tile.first) * ((in.nz + tile.second - 1) / tile.second);
      int prev = 0;
      // chunks for three quarters of a round of the CUs to five rounds, more
      // where those would be taller than a workgroup can address
      for (double rounds : {0.75, 1.0, 2.0, 3.0, 5.0}) {
        const long nch = std::max(1l, std::min((long)in.ny, (long)(rounds * cu_count) / cols));
        int h = temporal > 0 ? temporal : (int)((in.ny + nch - 1) / nch);
        if (h > sweep_max_height(in)) h = even_height(in.ny, sweep_max_height(in));
        if (h == prev) continue;
        prev = h;
        const SweepShape s = sweep_shape(in, tile.first, tile.second, h);
        double us = 0.0;
        for (long left = s.wgs; left > 0; left -= cu_count) us += s.at((double)std::min<long>(left, cu_count) / cu_count);
        if (s.wgs > cu_count) us *= SWEEP_ROUNDS;
        if (us < best) {
          best = us;
          shape[0] = s;
        }
      }
    }
    single += 2.0 * one_step_us(in);
    pair += best;
  } else {
    // every CU takes workgroups until none are left: the launch lasts as long
    // as their sum spread over the CUs, plus half of the longest at its end
    double best = 1e30;
    for (int cap : {4, 8, 16, 32, 64}) {
      std::vector<SweepShape> c(lats.size());
      double sum = 0.0, longest = 0.0;
      for (size_t i = 0; i < lats.size(); ++i) {
        const nflow_input& in = lats[i];
        const int h = even_height(in.ny, std::min(cap, sweep_max_height(in)));
        double least = 1e30;
        for (const auto& tile : sweep_tiles(in)) {
          const SweepShape s = sweep_shape(in, tile.first, tile.second, h);
          if (s.wgs * s.at(1.0) < least) {
            least = s.wgs * s.at(1.0);
            c[i] = s;
          }
        }
        sum += least;
        longest = std::max(longest, c[i].at(1.0));
      }
      const double us = (sum / cu_count + 0.5 * longest) * SWEEP_ROUNDS;
      if (us < best) {
        best = us;
        shape = c;
      }
    }
    for (const auto& in : lats) single += 2.0 * one_step_us(in);
    pair += best;
  }
  if (temporal < 0 && pair >= single) return none;
  return shape;
}

std::vector<SweepItem> sweep_work(const std::vector<nflow_input>& lats, const std::vector<SweepShape>& shape) {
  std::vector<SweepItem> out;
  if (shape.empty()) return out;
  // lattices of the longest workgroups first; each lattice's tiles in x, z, y
  // order, dealt so that the workgroups of an XCD (block id mod 8) hold
  // neighbouring tiles, which then share their halo in its L2
  std::vector<size_t> order(lats.size());
  for (size_t i = 0; i < order.size(); ++i) order[i] = i;
  std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) { return shape[a].at(1.0) > shape[b].at(1.0); });
  for (size_t i : order) {
    const SweepShape& s = shape[i];
    const nflow_input& in = lats[i];
    std::vector<SweepItem> items;
    for (int y = 0; y < in.ny; y += s.h)
      for (int z = 0; z < in.nz; z += s.tz)
        for (int x = 0; x < in.nx; x += s.tx) items.push_back(SweepItem{(int)i, x, z, y, s.tx, s.tz, s.h, 0});
    const size_t m = items.size(), len = (m + 7) / 8;
    for (size_t j = 0; j < len; ++j)
      for (size_t k = 0; k < 8; ++k) {
        const size_t at = m * k / 8 + j;
        out.push_back(at < m * (k + 1) / 8 ? items[at] : SweepItem{0, 0, 0, 0, 1, 1, 0, 0});
      }
  }
  return out;
}

}  // namespace nflow
