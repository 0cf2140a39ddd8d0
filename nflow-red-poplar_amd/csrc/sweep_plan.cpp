// sweep_plan.cpp -- tiles and chunk heights of two-step launches (k_sweep), and
// where they and launches of many steps (k_small) pay.
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
// start.  Fitted, with 4 us a launch and SWEEP_ROUNDS for more than one round
// of workgroups, to 600 launches of 62 cavities and channels of 40^3 to 512^3
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
static constexpr double SWEEP_ROUNDS = 1.06;

// Whether two steps in one launch beat two launches is a question of small
// lattices: chunks of few planes and CUs without work, where the estimate above
// is up to 7 us short for channels.  For that question alone: us of a workgroup
// of shape s when w of the CUs are busy, and us of two single steps.  Fitted,
// with 4 us for the launch, to 1,800 cavities and channels of 30,000 to 2,000,000
// nodes near the line (1.6 and 1.9 us rms, two single steps 5%).  On 800 others
// the answer costs 0.3% against the faster of the two, and 7 are more than 2%
// slower; by the estimate above 2.7%, and 142 were slower, by up to 40%, channels
// of some 100,000 nodes above all (274 x 28 x 24: 11.2 us a step, and 8.1 with
// one step per launch).
static double sweep_wg_us(const nflow_input& in, const SweepShape& s, double w) {
  const bool ch = in.casetype == NFLOW_CHANNEL;
  const double halo = ((s.tz < in.nz ? 2.0 * (s.tx + 2) : 0.0) + (s.tx < in.nx ? 2.0 * s.tz : 0.0)) / SWEEP_NT;
  const double fill = (double)s.tx * s.tz / SWEEP_NT * (in.nx % 32 ? 1.32 : 1.0);
  const double planes = (double)in.ny / ((in.ny - 1) / s.h + 1) + 0.28;
  const double plane = ch ? 4.84 + 0.39 * halo + 2.93 * w * fill - (s.tx < in.nx ? 0.18 : 0.0)
                          : 2.81 + 1.29 * halo + 3.16 * w * fill + (s.tx < in.nx ? 0.21 : 0.0);
  const double start = halo == 0.0 ? (ch ? 2.95 : 1.77) : ch ? 4.95 + 4.36 * halo : 2.97 + 4.59 * halo;
  return start + planes * plane;
}
static double two_steps_us(const nflow_input& in) {
  const bool ch = in.casetype == NFLOW_CHANNEL;
  return (double)in.nx * in.ny * in.nz / 39.0e3 * ((ch ? 2.05 : 2.0) + (in.nx % 32 ? 0.14 : 0.0));
}
static constexpr double SWEEP_LAUNCH_US = 4.0, TWO_LAUNCHES_US = 5.3;
// two steps per launch where they gain this much by the estimates
static constexpr double SWEEP_GAIN = 1.02;

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

static bool same_box(const nflow_input& a, const nflow_input& b) {
  return a.nx == b.nx && a.ny == b.ny && a.nz == b.nz && a.casetype == b.casetype;
}

std::vector<SweepShape> sweep_plan(const std::vector<nflow_input>& lats, int cu_count, int temporal) {
  std::vector<SweepShape> none;
  // a chunk height is a choice for one lattice; batches of several choose
  // for themselves or not at all
  if (temporal == 0 || lats.empty() || (temporal > 0 && lats.size() != 1)) return none;
  for (const auto& in : lats)
    if (in.casetype == NFLOW_PIPE || sweep_max_height(in) < std::max(temporal, 1)) return none;
  std::vector<SweepShape> shape(lats.size());
  double single = TWO_LAUNCHES_US, pair = SWEEP_LAUNCH_US;  // us of two steps, either way
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
    const long rounds = (shape[0].wgs - 1) / cu_count + 1;
    single += two_steps_us(in);
    // cavities in narrow rows, of which a launch holds every node at once (three
    // or, in rows on 128-byte lines, four workgroups of 256 a CU), take less
    // (64^3 7.0 us a step, 7.8 in pairs; 61 x 15 x 213 6.9 and 8.1)
    const bool lines = in.nx % 32 == 0;
    if (in.casetype == NFLOW_CAVITY && in.nx <= 192 &&
        (long long)in.nx * in.ny * in.nz <= (lines ? 1024ll : 768ll) * cu_count)
      single *= lines ? 0.83 : 0.9;
    pair += rounds * sweep_wg_us(in, shape[0], (double)shape[0].wgs / ((double)rounds * cu_count));
  } else {
    for (const auto& in : lats) single += two_steps_us(in);
    // a workgroup takes 1.77 + 1.28 x 2.81 us at least: many tiny lattices
    // need no search
    if (5.3 * lats.size() / cu_count >= single) return none;
    // every CU takes workgroups until none are left: the launch lasts as long
    // as their sum spread over the CUs, plus half of the longest at its end
    double best = 1e30;
    for (int cap : {4, 8, 16, 32, 64}) {
      std::vector<SweepShape> c(lats.size());
      double sum = 0.0, longest = 0.0;
      for (size_t i = 0; i < lats.size(); ++i) {
        const nflow_input& in = lats[i];
        if (i > 0 && same_box(in, lats[i - 1])) {
          c[i] = c[i - 1];
        } else {
          const int h = even_height(in.ny, std::min(cap, sweep_max_height(in)));
          double least = 1e30;
          for (const auto& tile : sweep_tiles(in)) {
            const SweepShape s = sweep_shape(in, tile.first, tile.second, h);
            if (s.wgs * s.at(1.0) < least) {
              least = s.wgs * s.at(1.0);
              c[i] = s;
            }
          }
        }
        sum += c[i].wgs * c[i].at(1.0);
        longest = std::max(longest, c[i].at(1.0));
      }
      const double us = (sum / cu_count + 0.5 * longest) * SWEEP_ROUNDS;
      if (us < best) {
        best = us;
        shape = c;
      }
    }
    // (35^3 x 57 channels: 105.5 us a step, and 78.6 with one step per launch)
    double sum = 0.0, longest = 0.0;
    for (size_t i = 0; i < lats.size(); ++i) {
      const double us = sweep_wg_us(lats[i], shape[i], 1.0);
      sum += shape[i].wgs * us;
      longest = std::max(longest, us);
    }
    pair += sum / cu_count + 0.5 * longest;
  }
  if (temporal < 0 && pair * SWEEP_GAIN >= single) return none;
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

// Each lattice keeps a CU to itself, 0.93 us a step however few its nodes, where
// one step per launch takes four lattices a CU and less time for fewer nodes: us
// per step of one step per launch / k_small, 4,096 lattices of 8 nodes 7.2 /
// 14.8, of 64 9.4 / 14.7, of 125 19.3 / 15.8, of 512 59 / 20; 2,048 of 64 4.9 /
// 7.4, 1,024 3.8 / 3.7.
int small_plan(const std::vector<nflow_input>& lats, int cu_count, int temporal) {
  if (temporal >= 0) return 0;
  long long most = 0, sum = 0;
  for (const auto& in : lats) {
    const long long n = (long long)in.nx * in.ny * in.nz;
    if (in.casetype != NFLOW_CAVITY || n > SMALL_NODES) return 0;
    most = std::max(most, n);
    sum += n;
  }
  const long long count = (long long)lats.size();
  return count > 4ll * cu_count && sum < 100 * count ? 0 : (int)most;
}

}  // namespace nflow
