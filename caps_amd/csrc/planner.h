// Plan choice when the caller passes no pattern (or mode CAPS_MODE_AUTO).
#pragma once
#include <string>

#include "../../include/caps_amd.h"

namespace caps {

// Workspace budget in bytes: the caller's (budget_set, capped at the free
// device memory) or, by default, half of the free device memory.
size_t planner_budget_bytes(long long budget_doubles, bool budget_set);

// One char per level: 'b' (batched) at every level whose workspace still fits
// the budget, 'd' below.  On one device a 'b' level only costs memory
// ((7/4)^levels growth), never communication, so batching is preferred.
std::string choose_pattern(const caps_desc &d, int mode, int moduli, long long budget_doubles,
                           bool budget_set);

// The pattern a plan runs for the requested one: recursive levels run batched,
// the deepest first, while they add at most the operands' own bytes (or
// any_bytes) to the requested pattern's workspace, but not more than
// extra_bytes, within limit_bytes.  The results do not depend on it.  items:
// problems of the same shape planned together.  An estimate (partials, exponents
// and alignment come on top): a plan that turns out larger than its limit is
// built again with drop_batched_level, one level less.
std::string batch_levels(const caps_desc &d, const std::string &pattern, int mode, int moduli,
                         int cutoff, size_t limit_bytes, size_t any_bytes, size_t extra_bytes,
                         int items = 1);
std::string drop_batched_level(const std::string &pattern, const std::string &run);
// the workspace that running `run` adds to the requested pattern's, as
// batch_levels estimates it
size_t batched_extra(const caps_desc &d, const std::string &pattern, const std::string &run,
                     int mode, int moduli, int cutoff);
inline bool has_recursive_level(const std::string &pattern) {
  return pattern.find_first_not_of("bB") != std::string::npos;
}
// any_bytes of one multiply with a workspace of its own (a 72nd of the device),
// and of a problem that shares the device with many or a scratch array
constexpr size_t BATCH_ANY_ALONE = (size_t)4 << 30;
constexpr size_t BATCH_ANY_SHARED = (size_t)64 << 20;
// what all cached plans together may add (a ninth of the device): 24 plans kept,
// each with 4 GiB, would hold a third of it for callers who asked for the
// smallest workspace
constexpr size_t BATCH_ANY_PLANS = (size_t)32 << 30;

// Leaf arithmetic when the caller asks for CAPS_MODE_AUTO.
int choose_mode(const caps_desc &d);

// The learned planner (tune_plan.cpp): false when no model is installed or no
// candidate is predicted to meet max_err.  pred (may be NULL) receives the
// model's predicted milliseconds and normwise error of the choice.
bool mlp_planner_choose(const caps_desc &d, int mask, double max_err, double spread, int &mode,
                        int &moduli, int &cutoff, std::string &pat, double *pred = nullptr);

// Uninstall m if it is the installed planner model (caps_mlp_destroy calls it).
void planner_forget_model(const caps_mlp *m);

}  // namespace caps
