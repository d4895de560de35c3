// How many workgroups should share one tile's work (a sweep's row tile, the backward's row or key
// tile) where the tiles alone leave the chip idle or uneven.  Host code.
#pragma once

#include <algorithm>

namespace fa4cp {

constexpr int kCus = 256;     // workgroups the chip runs at a time (one per CU)
constexpr int kMaxShares = 8;
constexpr float kOverUs = 11.5f;  // start and end of a workgroup
constexpr float kOverUs64 = 6.f;  // at head dim 64, beside another on the same CU

// Two classes of tiles, the long ones handed out first.  Work is counted in steps (key tiles,
// 32-row blocks) of `us` microseconds.
struct ShareLoad {
  int top;            // steps of the longest tile
  float avg;          // of the first class's average one
  int n;              // tiles of the first class
  int top2;           // the same of the second class (n2 = 0: none)
  float avg2;
  int n2;
  float us;           // microseconds per step
  float over = kOverUs;  // for the start and end of a workgroup
  float merge, read;  // merging k shares takes merge + k read microseconds,
  float slot = 0.f;   // and `slot` more for every share of the launch (written out and read by another)
  bool free2;         // the second class's shares are chosen apart (false: chunks as long as the first one's)
};

// What best_shares chose: at most k workgroups for a tile, about `chunk` steps each; of a tile of
// at most top2 steps k2, about chunk2 each.  k == 1: no tile is shared.
struct Shares {
  int k = 1, k2 = 1, chunk = 1, top2 = 0, chunk2 = 1;
};

// Workgroups that share a tile of n steps: the plan's rule and the kernels'.
constexpr int shares_of(int k, int chunk, int top2, int chunk2, int n) {
  const int c = n > top2 ? chunk : chunk2, m = (n + c - 1) / c;
  return m < 1 ? 1 : m > k ? k : m;
}

// The shares with the least estimated time, none unless they are 7 % faster.  A workgroup costs its steps
// plus `over`.
inline Shares best_shares(const ShareLoad& w, int most) {
  const float over = w.over / w.us;
  const float shortest = std::max(0.f, 2.f * w.avg - w.top);  // tile of the first class
  float one = 0.f, least = 0.f;
  Shares best;
  for (int k = 1; k <= most; ++k) {
    const int chunk = (w.top + k - 1) / k;
    const int tied = w.n2 ? std::max(1, std::min(k, (w.top2 + chunk - 1) / chunk)) : 1;
    for (int k2 = w.free2 ? 1 : tied; k2 <= (w.free2 && w.n2 ? k : tied); ++k2) {
      const float c1 = w.avg / k + over, c2 = w.avg2 / k2 + over;
      const int n1 = w.n * k, n2 = w.n2 * k2;
      const int q = n1 / kCus, r = n1 % kCus;
      // a last round that is not full costs a whole one where the tiles are equal; where they are not, the
      // short ones come last and even out.  (8832 tokens, H 32/8, fp16, cp 2, rank 1, the longest tile three
      // times the shortest: 340 us, in halves 387; 10720, H 16/16, D 256: 453, 545)
      const float even = n1 * c1 / kCus;
      const float longs = q == 0 ? (r > 0) * c1
                                 : even + ((q + (r > 0)) * c1 - even) * (shortest / k + over) / ((float)w.top / k + over);
      float t;
      if (n1 + n2 <= kCus) {
        t = std::max((float)w.top / k, (float)w.top2 / k2) + over;
      } else if (n2 == 0) {
        t = q < 3 ? longs : n1 * c1 / kCus + 0.5f * c1;
      } else {
        const int beside = (int)(c1 / c2) * (kCus - r);  // second-class workgroups that fit beside the last first-class ones
        t = n2 <= beside ? std::max(longs, q * c1 + (n2 + kCus - r - 1) / (kCus - r) * c2)
                         : std::max(longs, (n1 * c1 + n2 * c2) / kCus + 0.5f * c2);
      }
      t = std::max(t, (float)w.top / k + over);
      // The forward's tiles of both classes cut up, in more workgroups than CUs: 10-20 % over the estimate.
      // 13664 tokens (H 32/8, cp 8, rank 5): unshared 244 us, in halves 258; 16384: 287, 298; with a larger gain
      // ahead, 12288: 200, in 3 and 2 181.
      if (!w.free2 && k2 > 1 && n1 + n2 > kCus) t *= 1.2f;
      if (k > 1) t += (w.merge + w.read * k + w.slot * (n1 + n2)) / w.us;
      if (k == 1) one = least = t;
      else if (t < least) {
        least = t;
        best.k = k;
        best.k2 = k2;
      }
    }
  }
  if (least > 0.93f * one) return Shares{};
  best.chunk = (w.top + best.k - 1) / best.k;
  best.top2 = w.free2 && w.n2 ? w.top2 : 0;
  best.chunk2 = std::max(1, (w.top2 + best.k2 - 1) / best.k2);
  return best;
}

// The shares for the tiles of packed sequences, of one class: w.n tiles of w.avg steps on average and w.top
// the longest.  Their lengths differ and every CU takes the next one as it comes free, so the launch
// takes the chip's share of all steps and then about half a workgroup more, or one of the longest tile's.  (Above
// 0.8 workgroups a CU: some shader engines run out of CUs before others.)  None
// unless they are 7 % faster, nor where there are tiles enough to even out by themselves: 1.5 for a CU, 2 where
// two share one (15648 rows in three, H 8/2, cp 8, rank 6, 490 row tiles: 1425 us, in four 1540).
inline Shares packed_shares(const ShareLoad& w, int most) {
  if (2 * w.n > (w.over < kOverUs ? 4 : 3) * kCus) return Shares{};
  float one = 0.f, least = 0.f;
  Shares best;
  for (int k = 1; k <= most; ++k) {
    best.chunk = (w.top + k - 1) / k;
    const float k1 = k == 1 ? 1.f : std::max(1.f, std::min((float)k, w.avg / best.chunk + 0.5f));  // on average
    const float wgs = w.n * k1, each = w.avg / k1 * w.us + w.over;
    float t = wgs > 0.8f * kCus ? (w.n * w.avg * w.us + wgs * w.over) / kCus + 0.5f * each : each;
    t = std::max(t, w.top * w.us / k + w.over);
    if (k > 1) t += w.merge + w.read * k + w.slot * wgs;
    if (k == 1) one = least = t;
    else if (t < least) {
      least = t;
      best.k = k;
    }
  }
  if (least > 0.93f * one) return Shares{};
  best.chunk = (w.top + best.k - 1) / best.k;
  return best;
}

// Packed sequences: the share that the i-th of the ns workgroups of a head group's tile-th tile takes.  A short
// sequence's tiles have fewer than ns shares.  The XCDs, and in each its four shader engines, take the
// workgroups strictly in turn, so with the same i for share 0 of every tile an even ns leaves some of them
// without work (3, 4 and 5 shares forced on 210 drawn packed sweeps at head dim 128: 1.08, 1.24 and 1.20 of the
// unsplit time in the mean; turned, on 200 others, 1.08, 1.13 and 1.17).  Each term turns the tiles that the ones before it leave alike.
constexpr int turned_share(int i, int tile, int ns) {
  return (i + tile + (tile >> 1) + (tile >> 2) + (tile >> 3) + (tile >> 4)) % ns;
}

}  // namespace fa4cp
