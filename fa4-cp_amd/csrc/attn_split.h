// The split form of the fused sweep (attn_split.hip) as ring_sweep_launch uses it.
#pragma once

#include "attn_plan.h"
#include "common.h"

namespace fa4cp {

struct SweepParams;

// Workspace of a split sweep with n_hg head groups: split_words() counters that are zero between
// launches (rounded up to 256 bytes), the slots' outputs, then their LSEs (float32).
int64_t split_words(const SplitPlan& pl, int n_hg);
int64_t split_bytes(const SplitPlan& pl, int n_hg, int d);
// Queues the split sweep.
int launch_split(const SweepParams& p, const SplitPlan& pl, void* ws, int dtype, int d, int hp, bool paged,
                 hipStream_t st);

}  // namespace fa4cp
