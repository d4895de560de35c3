// The split form of the fused sweep (attn_split.hip) as ring_sweep_launch uses it.
#pragma once

#include "common.h"
#include "share_model.h"

namespace fa4cp {

struct SweepParams;

// How a sweep is split (see SweepSplit).
struct SplitPlan {
  Shares shares;
  int ns_back = 1, ns_front = 1, n_front = 0, n_row = 0, per_hg = 0;
  bool split() const { return shares.k > 1; }
};

// The plan for a sweep's shape (no pointer of `a` is followed).
SplitPlan split_plan(const fa4cp_sweep_args* a);
// Workspace of a split sweep with n_hg head groups: split_words() counters that are zero between
// launches (rounded up to 256 bytes), the slots' outputs, then their LSEs (float32).
int64_t split_words(const SplitPlan& pl, int n_hg);
int64_t split_bytes(const SplitPlan& pl, int n_hg, int d);
// Queues the split sweep.
int launch_split(const SweepParams& p, const SplitPlan& pl, void* ws, int dtype, int d, int hp, bool paged,
                 hipStream_t st);

}  // namespace fa4cp
