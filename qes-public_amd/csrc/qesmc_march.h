// The march (see qesmc_sor_fused.hip): what a launch is told of a problem and
// of the run, and its entry points for one problem and for a batch.
#pragma once

#include <vector>

#include "qesmc_internal.h"

namespace qesmc {

// One problem's arrays and tiles.
struct MarchItem {
  Dims d;
  int nq, nyt;  // x tiles, y tiles
  int ntiles;
  int first;            // its work-groups of the launch: ntiles from here
  float2 *set0, *set1;  // lambda, the two buffer sets
  const float2 *R;
  const unsigned *mask;
  const int *top;          // highest plane with a wall, per two rows and 32 pairs
  const unsigned *canon8;  // wall values per plane, 8 words (6 used)
  const float *sums;       // sum of the wall values each of the 64 masks selects, per plane
  unsigned *err;
  unsigned *status;
  unsigned *cur;                     // the set holding the latest iterate
  int begin[kMarchMaxSegments + 1];  // first plane of each segment (odd), then the end
};

// One launch.
struct MarchRun {
  float om[4];  // omega of each half-sweep (2T used)
  float tol;
  int t, itermax;
  int src;  // set this launch reads
  int fix;  // redo the last launch's first iteration if asked to (T = 1 only)
  // a batch: its problems, and the problem of each work-group
  const MarchItem *items;
  const int *which;
};

}  // namespace qesmc

void qesmc_march_item(const qesmc_ctx *x, const qesmc::MarchPlan &m, int first, qesmc::MarchItem &item);
int qesmc_march_batch_plan(qesmc_ctx *const *ctxs, int n, int T, std::vector<qesmc::MarchPlan> &plans,
                           double *expect_us);
hipError_t qesmc_launch_march_batch(hipStream_t s, int iters, int shape, int blocks, const qesmc::MarchRun &run);
hipError_t qesmc_march_settle_batch(hipStream_t s, const qesmc::MarchItem *items, int n, int hi, float tol);
