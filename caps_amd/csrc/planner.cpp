// Greedy BFS/DFS choice under a memory budget.  The reference's automatic
// rule (multiply.cpp:43-66 with enoughMemory, memory.cpp:22-29) takes a BFS
// step only while the workspace it needs fits the budget set by
// setAvailableMemory (memory.cpp:31-33; drivers pass -m / -k,
// randombenchmark.cpp:45-48), and only with several processes.  On one device
// a 'b' level is batching, limited by workspace alone, so the same budget
// decides it: a level becomes 'b' when the whole plan's device workspace still
// fits.
#include "planner.h"

#include <hip/hip_runtime.h>

#include <algorithm>

#include "engine.h"

namespace caps {

size_t planner_budget_bytes(long long budget_doubles, bool budget_set) {
  size_t freeb = 0, totalb = 0;
  const bool have_free = hipMemGetInfo(&freeb, &totalb) == hipSuccess;
  if (budget_set) {
    // the caller's budget, capped at what the device has free
    size_t b = (size_t)budget_doubles * sizeof(double);
    return have_free && b > freeb ? freeb : b;
  }
  // no budget set: half of the free device memory (the reference's default
  // of 2^28 doubles, memory.cpp:4, when no device answers)
  return have_free ? freeb / 2 : (size_t)(1LL << 28) * sizeof(double);
}

std::string choose_pattern(const caps_desc &d, int mode, int moduli, long long budget_doubles,
                           bool budget_set) {
  std::string pat((size_t)d.nrec, 'd');
  const size_t budget = planner_budget_bytes(budget_doubles, budget_set);
  for (int l = 0; l < d.nrec; l++) {
    std::string trial = pat;
    trial[(size_t)l] = 'b';
    if (plan_workspace_bytes(d, trial, mode, moduli, 0) <= budget) pat = trial;
  }
  return pat;
}

namespace {

// Workspace of one problem, from the sizes alone: per level and sub-problem
// 15 half-size matrices batched or 2 recursive, and what the leaves of the
// bottom batch need.
double workspace_estimate(const caps_desc &d, const std::string &pattern, int mode, int moduli,
                          int cutoff) {
  const bool residue = residue_mode(mode);
  const int m0 = d.lda >> d.nrec;
  auto bytes = [&](int s) {  // one s x s matrix
    const double leaves = (double)(s / m0) * (s / m0);
    return residue ? leaves * residue_area(m0) * moduli : 8.0 * s * s;
  };
  double w = residue ? 3 * bytes(d.lda) : 0.0, batch = 1;
  int s = d.lda;
  for (int l = 0; l < d.nrec - cutoff; l++) {
    s /= 2;
    const bool b = pattern[(size_t)l] == 'b' || pattern[(size_t)l] == 'B';
    w += batch * bytes(s) * (b ? 15 : 2);
    if (b) batch *= 7;
  }
  if (!residue && d.bs != 1 && d.bs != m0) w += 3 * batch * bytes(s);  // column-major leaves
  if (mode == CAPS_MODE_OZAKI_INT8) w += 3.0 * batch * residue_area(s) * moduli;
  return w;
}

}  // namespace

// A 'd' level multiplies its seven products one after another to keep its
// workspace at two half-size matrices.  On this device that leaves small
// products alone on 256 CUs and costs 13 dependent launches per level, while
// 288 GB hold far more than the operands; BFS and DFS steps evaluate the same
// expression trees.  Measured (FP64): n = 4096 'ddd' 7.42 ms recursive, 2.07
// ms with its two lower levels batched, 1.78 with all three (2 GB); n = 392
// 'bdd' 563 and 47 us.
std::string batch_levels(const caps_desc &d, const std::string &pattern, int mode, int moduli,
                         int cutoff, size_t limit_bytes, size_t any_bytes, size_t extra_bytes,
                         int items) {
  std::string run = pattern;
  // a launch takes at most 65,535 leaves of the leaf-only split (grid.y)
  double batch = items;
  for (int l = 0; l < d.nrec - cutoff; l++)
    if (pattern[(size_t)l] == 'b' || pattern[(size_t)l] == 'B') batch *= 7;
  const double extra =
      std::min(std::max(24.0 * d.lda * d.lda, (double)any_bytes), (double)extra_bytes);
  const double limit = std::min(workspace_estimate(d, pattern, mode, moduli, cutoff) + extra,
                                (double)limit_bytes);
  for (int l = d.nrec - cutoff - 1; l >= 0; l--) {
    if (run[(size_t)l] == 'b' || run[(size_t)l] == 'B') continue;
    std::string trial = run;
    trial[(size_t)l] = 'b';
    if (7 * batch > 65535 || workspace_estimate(d, trial, mode, moduli, cutoff) > limit) continue;
    run = trial;
    batch *= 7;
  }
  return run;
}

std::string drop_batched_level(const std::string &pattern, const std::string &run) {
  std::string r = run;  // the last one that batch_levels took: the outermost
  for (size_t l = 0; l < r.size(); l++)
    if (r[l] != pattern[l]) {
      r[l] = pattern[l];
      break;
    }
  return r;
}

size_t batched_extra(const caps_desc &d, const std::string &pattern, const std::string &run,
                     int mode, int moduli, int cutoff) {
  return (size_t)(workspace_estimate(d, run, mode, moduli, cutoff) -
                  workspace_estimate(d, pattern, mode, moduli, cutoff));
}

int choose_mode(const caps_desc &) { return CAPS_MODE_FP64; }

}  // namespace caps
