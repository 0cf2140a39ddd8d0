// sweep_plan.hpp -- which lattices take two steps per launch (k_sweep), in
// which tiles and chunks of planes, and which many (k_small).  Host code
// without HIP.
#pragma once
#include <vector>

#include "nflow.h"

namespace nflow {

// Work of one workgroup of k_sweep (two steps per launch): a tile of tx x tz
// nodes of the x-z plane from (x0, z0), one per thread (tx tz <= SWEEP_NT, tz
// <= SWEEP_ROWS), swept over the y planes [ya, ya + h); h = 0: no work.  The
// exchange between the columns holds, per crossing population, SWEEP_SLOT0
// elements where e_z = 0, at least tz (tx + 2), and SWEEP_SLOT1 where it is
// not, at least (tz + 1) (tx + 2); two planes of it fill the LDS.
enum : int { SWEEP_NT = 1024, SWEEP_ROWS = 32, SWEEP_SLOT0 = 1088, SWEEP_SLOT1 = 1296 };
struct alignas(16) SweepItem {
  int lat, x0, z0, ya, tx, tz, h, pad;
};

// A lattice's tiles (all of one shape but the last in x and in z) and chunk
// height, with its estimated work: workgroups, and us of each when w (0 to 1)
// of the CUs are busy.
struct SweepShape {
  int tx = 0, tz = 0, h = 0;
  long wgs = 0;
  double us0 = 0.0, us1 = 0.0;  // us0 + w us1
  double at(double w) const { return us0 + w * us1; }
};

// The tallest chunk of planes of a lattice whose window a workgroup can
// address; 0: none.
int sweep_max_height(const nflow_input& in);

// Two steps per launch for FP32 cavity and channel lattices without solid
// nodes (a pipe has them: none): one shape per lattice, or none where one step
// per launch is to be used.  temporal: nflow_tuning's.
std::vector<SweepShape> sweep_plan(const std::vector<nflow_input>& lats, int cu_count, int temporal);

// The work list of a plan.
std::vector<SweepItem> sweep_work(const std::vector<nflow_input>& lats, const std::vector<SweepShape>& plan);

// k_small: whole lattices of up to SMALL_NODES nodes in a workgroup's LDS.  One
// compute unit's work per step meets the launch it saves near 2,000 nodes: us
// per step of one step per launch / k_small, MRT, 512 nodes 3.8 / 1.2, 1000 4.0
// / 1.75, 1100 4.0 / 2.3, 1728 4.1 / 3.1, 2028 4.1 / 3.8, 2048 in a row 3.65 /
// 3.8.
enum : int { SMALL_NT = 1024, SMALL_NODES = 1920 };

// Many steps per launch for FP32 cavities without solid nodes: the nodes of the
// largest where all are to run in k_small, else 0.
int small_plan(const std::vector<nflow_input>& lats, int cu_count, int temporal);

}  // namespace nflow
