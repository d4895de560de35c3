// Plans of the attention launches: which build of a kernel runs and how many workgroups share a
// tile.  Host code without HIP, so that a plan can be looked at where there is no GPU.
#pragma once

#include <stdint.h>

#include <algorithm>

#include "../../include/fa4cp.h"
#include "share_model.h"

namespace fa4cp {

// Heads of one kv-head group that a workgroup takes (HP of the kernels).
inline int heads_per_wg(int group) {
  if (group % 4 == 0) return 4;
  if (group % 2 == 0) return 2;
  return 1;
}

constexpr int kPPWaves = 8;  // wavefronts of a ping-pong kernel's workgroup, 32 (row, head) pairs each

// Workgroups per CU that the 16-bit pipeline's kernels are built for (their WGS).  At head dim 64 the
// LDS tiles take 57 KB and the registers fit 128 without a spill, so two can run on a CU, one's loads,
// softmax, start and end beside the other's MFMAs.  Sweeps (GPU time, the V^T launch with them): 131072 tokens (H
// 32/8, cp 8, rank 3) 9000 -> 8325 us, 49152 (cp 4, rank 2) 2555 -> 2390, 24 short sequences of 16 heads 58.4 ->
// 52.6.  Either of two on a CU takes 1.85 times as long, so there must be more than that:
// * more than two for each CU: with fewer all start at once, the longest two to a CU while others fall idle (432 row
//   tiles, H 24/8, 4504 rows, cp 8, rank 0: 800 us one per CU, 1170 two).  Two by one per CU, in the mean of drawn
//   shapes of 257-512 row tiles and of more: one sequence 1.14 (34), 0.97 (62); packed 1.07 (20), 0.97 (51); per-step
//   1.06 (20), 0.96 (25);
// * in a sweep of fewer than four head groups, whose row tiles several XCDs share, four for each (512-1024 row
//   tiles 1.03 (12; 27782 rows of H 8/1, cp 4, rank 2: 3650 and 4130 us), packed 1.10 (4), more 0.96 (3));
// * more than one for each where all row tiles are short (few_rows) and their start and end count for more: 0.93 (63;
//   H 144/144, cp 2, 296 rows, 288 row tiles: 52 and 45 us), with fewer 1.03 (12);
// * or where the sweep is split, in workgroups of about equal length: 0.91-0.94 (39).
inline bool two_per_cu(int d, int64_t workgroups, int most_alone) { return d == 64 && workgroups > most_alone; }
inline bool few_rows(int64_t longest, int rows) { return longest <= std::min(4 * rows, 512); }

// Row tiles of `rows` rows, at most n_rt in a sequence, that nseq sequences of `total` rows in all make.
// Only the device knows the lengths of packed ones: about half a tile per sequence more than
// total / rows.  (A grid of n_rt tiles for each of nine sequences of 1024 rows in all, the longest 350, H
// 32/8, has 432 workgroups, 160 of them with rows.)
inline int64_t working_row_tiles(int64_t total, int rows, int nseq, int64_t n_rt) {
  return nseq > 1 ? std::min(nseq * n_rt, total / rows + nseq / 2) : n_rt;
}

// The build of the unsplit sweep, whose workgroups without rows come last.
inline bool sweep_two_per_cu(const fa4cp_sweep_args* a) {
  const int hp = heads_per_wg(a->h_q / a->h_kv), rows = 32 * kPPWaves / hp;
  const int longest = a->cu ? a->max_seqlen : a->total;
  const int64_t n_rt = ((int64_t)longest + rows - 1) / rows;
  const int n_hg = a->h_q / hp;
  return two_per_cu(a->d, n_hg * working_row_tiles(a->total, rows, a->cu ? a->nseq : 1, n_rt),
                    few_rows(longest, rows) ? kCus : n_hg < 4 ? 4 * kCus : 2 * kCus);
}

// The build of the V^T kernel for one attention call.  Its workgroups without rows stand among the others
// and hold up their start: where all row tiles are short the grid counts (attention of two steps, the grid above
// 256 workgroups, those with rows below: two per CU 0.93 of the time in the mean of 18 shapes; nine sequences of 784
// rows, H 32/8, 44 and 38 us), elsewhere the workgroups with rows (1.05 in the mean of 42; the nine sequences above
// 43.1 and 47.4 us, 7652 rows in three, H 8/1, 130 and 147).
inline bool attn_two_per_cu(const fa4cp_attn_args* a) {
  const int hp = heads_per_wg(a->h_q / a->h_kv), rows = 32 * kPPWaves / hp, nseq = a->cu_q ? a->nseq : 1;
  const bool all = a->q_sel == FA4CP_SEL_ALL;
  auto selected = [&](int n) { return all ? n : (n + 1) / 2; };
  const int longest = selected(a->cu_q ? a->max_seqlen_q : a->total_q);
  const int64_t n_rt = ((int64_t)longest + rows - 1) / rows;
  const bool few = few_rows(longest, rows);
  const int64_t tiles = few ? nseq * n_rt : working_row_tiles(selected(a->total_q), rows, nseq, n_rt);
  return two_per_cu(a->d, a->h_q / hp * tiles, few ? kCus : 2 * kCus);
}

// How a sweep is split (see SweepSplit in attn_split.hip).
struct SplitPlan {
  Shares shares;
  int ns_back = 1, ns_front = 1, n_front = 0, n_row = 0, per_hg = 0;
  bool split() const { return shares.k > 1; }
};

// The length whose tiles stand for those of packed sequences of `total` rows in all: the longer ones
// hold more of the rows than their number says.
inline int mixed_len(int total, int nseq, int longest) {
  return (int)((std::max(1, total / nseq) + 2 * (int64_t)longest) / 3);
}

// Slots of one launch: of a sweep 256 rows of float32 outputs and their LSEs each (129 KB at head dim 128, 257 at
// 256: 514 MB at most), of the backward 128 KB (dq; 256 MB).  Half as many would take the gain from long
// sweeps of few heads at head dim 256 (74752 tokens, H 8/2, cp 8, rank 7: 3242 us unsplit, in four 2554 with 299
// MB; 143008 tokens: 9941, in three 8705 with 431).
constexpr int kMaxSlots = 2048;
constexpr float kSlotUs = 0.035f;  // a slot of 128 KB written and read while the chip is full of workgroups

// The plan for a sweep's shape (no pointer of `a` is followed).
// The number of shares comes from best_shares' estimate: the row tiles that meet the later sources
// (about `avg` key tiles each) before the others, 1.65 us a key tile (1 us at head dim 64), a merge
// of 5 us plus 1.25 us per share and 128 columns, and at head dim 128 kSlotUs for every share of the launch (at
// 64, half the bytes and two workgroups on a CU, it hides).  Some of the shapes it was set by (one
// and four rings, D 64 / 128 / 256, 16 to 512 row tiles; GPU time, us):
//   shares                                1     2     3     4     6     8
//   2048 tokens, H 8/2, cp 4, rank 1     52    42    39    38    38    40   (chosen: 6)
//   8192, H 32/8, cp 8, rank 3          144    96    88   107   103   116   (3)
//   16384, rank 3                       298   282   270   298   298   313   (3)
//   16384, rank 7 (equal row tiles)     264   267   277   291   319   344   (1)
//   24576, rank 3                       555   573   560   623   594   626   (1)
//   8832, fp16, cp 2, rank 1            340   387                            (1)
//   8192, e4m3, rank 3                  113    80    69    85    84   100   (3)
//   16384, H 16/2, D 256, rank 3        476   301   278   353   335   400   (3)
// Packed sequences go by packed_shares.  By best_shares, with two classes of row tiles from an average
// sequence, 27 of 210 drawn shapes at head dim 128 were more than 5 % slower than unsplit (30 sequences of 7708 rows, H
// 8/1, e4m3, cp 4, rank 1: 74 us, in four 129).  Time by the unsplit one's, mean and worst of 90 shapes that either
// splits, and with packed_shares and turned_share: head dim 128 0.89 (1.32), 0.84 (1.06); 64 0.76 (1.25), 0.76 (1.12);
// 256 0.94 (1.48), 0.82 (1.09).
// At head dim 256 a share costs more: the merging workgroup takes 10 us and 8 for each (its 256 KB come one load
// at a time: beside the 128 registers of the output there is room for no more), and the launch 0.1 us for
// each (256 KB written and read at the copy rate).  At 2.5 us and nothing, shapes were split that are
// faster whole or in fewer shares (us unsplit, in the shares chosen then, and now):
//   1024 tokens, H 8/2, fp16, cp 2, rank 1        52   72 (4)   52 (1)
//   8000, H 32/8, bf16, cp 4, rank 3             261  292 (2)  261 (1)
//   8772, H 32/8, e4m3, cp 2, rank 1             340  449 (2)  340 (1)
//   1456, H 16/2, fp16, cp 8, rank 3              69   82 (5)   70 (3)
//   2368, H 8/2, bf16, cp 8, rank 5               85   98 (7)   77 (3)
//   nine sequences, 7888, H 16/2, cp 8, rank 6    84  108 (6)   77 (2)
inline SplitPlan split_plan(const fa4cp_sweep_args* a) {
  constexpr int kMaxRowTiles = 1024;
  SplitPlan pl;
  const bool fp8 = a->dtype == FA4CP_E4M3;
  const int bn = fp8 ? (a->d == 256 ? 64 : 128) : (a->d == 256 ? 32 : 64);
  const int hp = heads_per_wg(a->h_q / a->h_kv), rows = 32 * kPPWaves / hp;
  const int n_hg = a->h_q / hp;
  const int nseq = a->cu ? a->nseq : 1;
  const int longest = a->cu ? std::min(a->max_seqlen, a->total) : a->total;
  if (longest <= 0) return pl;
  const int64_t n_rt = (longest + rows - 1) / rows;
  // packed: at most one row tile per sequence beyond total / rows
  const int64_t n_row = nseq > 1 ? std::min(nseq * n_rt, (int64_t)a->total / rows + nseq) : n_rt;
  if (n_hg * n_row > kMaxRowTiles) return pl;
  auto tiles = [&](int keys) { return (keys + bn - 1) / bn; };
  const int late_steps = a->cp_size - 1 - a->cp_rank;
  // key tiles of row tile rt of a sequence of L rows
  auto cost = [&](int L, int rt, bool back) {
    return (std::min((rt + 1) * rows, L) - 1) / bn + 1 + a->cp_rank * tiles(L / 2) + (back ? late_steps * tiles(L) : 0);
  };
  // the classes of row tiles, of one sequence for all when packed
  const int L = nseq > 1 ? mixed_len(a->total, nseq, longest) : longest;
  const int rts = (L + rows - 1) / rows;
  const int fronts = late_steps > 0 ? (L / 2) / rows : 0;
  const int top = cost(longest, (int)n_rt - 1, true);
  if (top > 1 << 20) return pl;
  const int front_top = fronts ? cost(L, fronts - 1, false) : 0;
  ShareLoad w;
  w.top = top;
  w.avg = 0.5f * (cost(L, rts - 1, true) + cost(L, fronts, true));
  w.n = n_hg * (rts - fronts);
  w.top2 = front_top;
  w.avg2 = fronts ? 0.5f * (front_top + cost(L, 0, false)) : 0.f;
  w.n2 = n_hg * fronts;
  w.us = a->d == 64 ? 1.f : 1.65f;
  const bool wide = a->d == 256;
  w.merge = wide ? 10.f : 5.f;
  w.read = wide ? 8.f : 1.25f * a->d / 128.f;
  w.slot = wide ? 0.1f : a->d == 128 ? kSlotUs : 0.f;
  w.free2 = false;
  // (per_hg, the slots of a head group, is rounded up to 8)
  int most = std::min(kMaxShares, kMaxSlots / (int)(n_hg * n_row));
  while (most > 1 && n_hg * ((n_row * most + 7) / 8 * 8) > kMaxSlots) --most;
  if (nseq > 1) {
    w.avg = ((rts - fronts) * w.avg + fronts * w.avg2) / rts;
    w.n = n_hg * (int)std::max<int64_t>(1, working_row_tiles(a->total, rows, nseq, n_rt));
    if (a->d == 64) w.over = kOverUs64;
    pl.shares = packed_shares(w, most);
  } else {
    pl.shares = best_shares(w, most);
  }
  if (pl.shares.k == 1) return pl;
  pl.n_row = (int)n_row;
  pl.ns_back = pl.shares.k;
  if (nseq == 1 && fronts > 0) {
    pl.n_front = fronts;
    pl.ns_front = pl.shares.k2;
  }
  pl.per_hg = ((pl.n_row - pl.n_front) * pl.ns_back + pl.n_front * pl.ns_front + 7) / 8 * 8;
  return pl;
}

constexpr int kBwdRows = 32;  // query rows (dq) or keys (dk/dv) per wavefront
constexpr int kDkdvKeys = 4 * kBwdRows;  // keys per dk/dv workgroup

// The 32-row blocks that hold rows [row, L) of a sequence of L: the first one's first row, and how many.
// A key tile walks them, with row the first of its keys' causal rows, or the back half's first.
constexpr int first_block_row(int row) { return row / kBwdRows * kBwdRows; }
constexpr int row_blocks(int L, int row) { return (L - first_block_row(row) + kBwdRows - 1) / kBwdRows; }

// Tiles of the two gradient kernels and the workgroups that share one.
struct BwdPlan {
  int64_t dq_tiles = 0, kv_tiles = 0;
  int dq_rows = 0;  // rows of a dq tile
  Shares dq, kv;
};

// A 32-key block of dq takes 1.2 us and a 32-row block of dk / dv 1.02 (measured, head dim 128, the
// chip full; dq at 256, half the rows, 1.7).  dq's row tiles are shared wherever best_shares finds it faster (backward, GPU time in
// us, shares of the back-half / other row tiles: 8192 tokens, H 32/8, cp 4, rank 1: none 622, 2/1 584,
// 2/2 564 (chosen), 3/2 589; 16384, cp 8, rank 3: 1098, 1046, 1000 (chosen), 1054; rank 7, equal row
// tiles: 985 (chosen), 1071, 992, 1050).  dk / dv's key tiles only where all shares run at once: the
// workgroups stream the query blocks in step, and shares at other blocks cost more in L2
// misses than the even split gains (8192 tokens: none 622, two shares 628-651, three 634-650; 24576
// tokens, H 16/2: 1311, 1337-1389), but 32 key tiles leave the chip idle (2048 tokens, H 8/2: 138,
// 120, 113; four 112).  At head dim 256 a block takes the MFMAs twice as long and the even split wins up to
// 256 tiles, of up to four times as many shares as CUs (backward: 16384 tokens, H 16/2, cp 8, rank 3, 256 tiles
// 1333 and 1165; 8192, cp 4, 128 tiles: two shares 727, up to eight 610; four sequences, H 8/2, 273 and 205),
// not beyond (32768 tokens, cp 4, 512 tiles 8450 and 8559).  There a share costs 0.08 us for its 256 KB (without
// that, 3072 tokens, H 24/8, cp 8, rank 6, short tiles: unshared 266, shared 281).
inline BwdPlan bwd_plan(const fa4cp_sweep_bwd_args& a) {
  constexpr int kMaxTiles = 1024;
  BwdPlan pl;
  const int group = a.h_q / a.h_kv, nseq = a.cu ? a.nseq : 1;
  const int hp = group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
  const int longest = a.cu ? std::min(a.max_seqlen, a.total) : a.total;
  const int rows = a.d == 256 ? kBwdRows : kBwdRows * 2 * (4 / hp);
  const int64_t row_tiles = (longest + rows - 1) / rows, key_tiles = (longest + kDkdvKeys - 1) / kDkdvKeys;
  pl.dq_rows = rows;
  pl.dq_tiles = nseq * row_tiles * (a.h_q / hp);
  pl.kv_tiles = (int64_t)a.cp_size * a.h_kv * nseq * key_tiles;
  if (longest <= 0) return pl;
  const int L = nseq > 1 ? mixed_len(a.total, nseq, longest) : longest;
  const int late = a.cp_size - 1 - a.cp_rank;
  auto blocks = [](int n) { return (n + kBwdRows - 1) / kBwdRows; };
  if (pl.dq_tiles <= kMaxTiles) {
    auto cost = [&](int len, int rt, bool back) {
      return blocks(std::min((rt + 1) * rows, len)) + a.cp_rank * blocks(len / 2) + (back ? late * blocks(len) : 0);
    };
    const int rts = (L + rows - 1) / rows, fronts = late > 0 ? L / 2 / rows : 0;
    ShareLoad w;
    w.top = cost(longest, (int)row_tiles - 1, true);
    w.avg = 0.5f * (cost(L, rts - 1, true) + cost(L, fronts, true));
    w.n = (a.h_q / hp) * (rts - fronts);
    w.top2 = fronts ? cost(L, fronts - 1, false) : 0;
    w.avg2 = fronts ? 0.5f * (w.top2 + cost(L, 0, false)) : 0.f;
    w.n2 = (a.h_q / hp) * fronts;
    w.us = a.d == 256 ? 1.7f : 1.2f * a.d / 128.f;
    w.merge = 5.f;
    w.read = 1.25f * a.d / 128.f;
    w.free2 = true;
    const int most = std::min<int64_t>(kMaxShares, kMaxSlots / pl.dq_tiles);
    if (nseq > 1) {
      w.avg = ((rts - fronts) * w.avg + fronts * w.avg2) / rts;
      w.n = a.h_q / hp * (int)std::max<int64_t>(1, working_row_tiles(a.total, rows, nseq, row_tiles));
      w.slot = a.d == 64 ? 0.f : kSlotUs;  // (128 KB at head dim 256 too)
      if (a.d == 64) w.over = kOverUs64;
      pl.dq = packed_shares(w, most);
    } else {
      pl.dq = best_shares(w, most);
    }
  }
  const bool wide = a.d == 256;
  if (2 * pl.kv_tiles <= (wide ? 2 : 1) * kCus) {
    // earlier sources: every row, the front half of the keys; own: half of the rows on average; later
    // sources: the back-half rows.  The own tiles of more blocks than a later source's are of the first
    // class (about three quarters of the rows; the first half of the tiles, short of a middle one as long as a later source's).
    const int all = row_blocks(L, 0) * group, back = row_blocks(L, L / 2) * group;
    const int kts = (L + kDkdvKeys - 1) / kDkdvKeys, early = a.cp_rank * ((L / 2 + kDkdvKeys - 1) / kDkdvKeys);
    int own1 = 0;
    while (own1 < kts && row_blocks(L, own1 * kDkdvKeys) * group > back) ++own1;
    ShareLoad w;
    w.top = blocks(longest) * group;
    if (back < all) {
      w.n = a.h_kv * (early + own1);
      w.avg = all * (early + 0.75f * own1) / (early + own1);
      w.top2 = back;
      w.n2 = a.h_kv * (late * kts + kts - own1);
      w.avg2 = w.n2 ? ((float)back * late * kts + 0.25f * all * (kts - own1)) / (late * kts + kts - own1) : 0.f;
    } else {  // a single key tile of few rows: all alike
      w.n = a.h_kv * (early + kts + late * kts);
      w.avg = all;
      w.top2 = w.n2 = 0;
      w.avg2 = 0.f;
    }
    w.us = wide ? 1.75f : 1.02f * a.d / 128.f;
    w.merge = wide ? 6.f : 5.f;
    w.read = wide ? 0.f : 1.25f * a.d / 128.f;
    w.slot = wide ? 0.08f : 0.f;  // 256 KB each
    w.free2 = true;
    const int most = std::min<int64_t>(kMaxShares, (wide ? 4 : 1) * kCus / pl.kv_tiles);
    if (nseq > 1) {
      w.avg = (w.n * w.avg + w.n2 * w.avg2) / (w.n + w.n2);
      w.n = std::max(1, (int)((float)a.total / L * (w.n + w.n2)));
      if (a.d == 128) w.slot = kSlotUs;
      pl.kv = packed_shares(w, most);
    } else {
      pl.kv = best_shares(w, most);
    }
  }
  return pl;
}

}  // namespace fa4cp
