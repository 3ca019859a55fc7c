// Host plan of the prefill kernel (prefill_kernel.h) and the numbering of its workgroups: plain C++, so that
// tests/prefill_plan_check.cpp can enumerate every launch the plans can make.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>

#include "limits.h"

namespace kvq {

constexpr int kPT = 64;       // keys per tile
constexpr int kPRows = 256;   // query rows per workgroup (8 waves x 32 MFMA columns)
constexpr int kPTargetWgs = 256;  // one workgroup per CU

struct PrePlan {
  int nbk, rowblocks, nunits, nsplit, tiles, chunk;
  bool unequal;       // row blocks of unequal length, to be run from the longest down
  int longest_first;  // how (see prefill_wg)
};

// Splits merged by the last of them to arrive; more take prefill_combine_kernel. Few splits are cheaper
// in the kernel (the last 512-token chunk of 16384, 4 splits: 155.2 against 161.3 us for the layer
// step), many in a launch of their own, whose loads run side by side: 64 rows of 4 KV heads over 8192
// keys (32 splits) 45.5 -> 18.4 us, over 32768 (64 splits) 81.2 -> 28.0.
constexpr int kPFusedMaxSplit = 4;

// Cut `pl` into `nsplit` splits. What follows from the count is set here and nowhere else, so that every plan is
// numbered for the count it runs with.
inline void set_splits(PrePlan* pl, int nsplit) {
  pl->nsplit = nsplit;
  pl->chunk = (pl->tiles + nsplit - 1) / nsplit * kPT;
  const bool dealt = pl->nbk % kXcds == 0 || (pl->nbk < kXcds && kXcds % pl->nbk == 0 &&
                                              (int64_t)pl->rowblocks * nsplit % (kXcds / pl->nbk) == 0);
  pl->longest_first = !pl->unequal ? 0 : dealt ? 1 : 2;
}

inline PrePlan prefill_plan(int B, int Hq, int Hkv, int L, int S, int window, int causal) {
  PrePlan pl;
  const int rep = Hq / Hkv, nrows = rep * L;
  pl.nbk = B * Hkv;
  pl.rowblocks = (nrows + kPRows - 1) / kPRows;
  pl.nunits = pl.nbk * pl.rowblocks;
  // keys a row block sees: the whole context, or about a window; the first row block of a causal call
  const int span = window > 0 ? std::min(S, window + kPRows) : S;
  const int first = causal && window == 0 ? std::min(S, S - L + (kPRows + rep - 1) / rep) : span;
  const int tiles = (span + kPT - 1) / kPT, tiles0 = (first + kPT - 1) / kPT;
  pl.tiles = tiles;
  pl.unequal = 2 * tiles0 <= tiles;
  int ns = (kPTargetWgs + pl.nunits - 1) / pl.nunits;
  if (pl.unequal) {
    // A causal prompt, whose first row blocks see few keys: the number of splits with the shortest
    // estimate, in tiles (of about 2.2 us at 128 dims), of max(the longest workgroup, an even share of
    // all work), a workgroup costing 4 tiles besides its own and 2 more where it takes part in a merge.
    // 32 KV heads of 96 dims, 1999 tokens, 1 / 2 splits: 56 / 48 us; 4 KV heads of 8 query heads of
    // 128 dims, 1000 tokens, 2 / 3 / 4 splits: 26.5 / 24.8 / 37.9 us.
    const float avg = 0.5f * (tiles + tiles0);
    float best = 0.0f;
    for (int c = 1; c <= kPFusedMaxSplit; ++c) {
      const int chunk = (tiles + c - 1) / c, cost = c > 1 ? 6 : 4;
      const float total = pl.nunits * (avg + (avg / chunk + 0.5f) * cost);
      const float est = std::max(total / kPTargetWgs, (float)(chunk + cost));
      if (c == 1 || est < best) {
        best = est;
        ns = c;
      }
    }
  }
  ns = std::min(ns, std::max(1, tiles / 4));  // at least about 4 tiles per split
  set_splits(&pl, pl.nunits > kMaxCountedUnits ? 1 : std::max(1, std::min(ns, kMaxSplit)));
  return pl;
}

// Workspace: [arrival counters (the block shared with decode)][o partials][(m, l) partials]
struct PreLayout {
  size_t o, ml, total;
};
inline PreLayout prefill_layout(const PrePlan& pl, int D, bool f32_partials) {
  PreLayout l;
  const size_t slots = (size_t)pl.nunits * pl.nsplit * kPRows;
  l.o = kCounterBytes;
  l.ml = l.o + slots * D * (f32_partials ? sizeof(float) : sizeof(uint16_t));
  // records: (m, l), or (m, l, 2^e, -) of an fp16 row
  l.total = l.ml + (slots * (f32_partials ? 2 : 4) * sizeof(float) + 255) / 256 * 256;
  return l;
}

// Workgroup `wg` of the launch's `grid` = nbk rowblocks nsplit: its (sequence, KV head) pair, row block and
// split, each combination once. The row blocks of one (pair, split) share every K/V tile, so they are
// consecutive, and consecutive workgroups are placed on one XCD (the hardware hands workgroups to the 8
// XCDs in turn; xcd_remap: the grid is a multiple of 8): each tile is fetched into one L2 rather than eight.
struct PreWg {
  int bk, rb, split;
};
constexpr PreWg prefill_wg(int wg, int grid, int rowblocks, int nsplit, int xcd_remap, int longest_first) {
  PreWg w{};
  if (longest_first == 1) {
    // a causal prompt, whose last row blocks see many times the keys of its first: every XCD takes its
    // share of the pairs (or a pair's row blocks are dealt to several XCDs, whose number then divides
    // rowblocks nsplit: set_splits) and runs the row blocks of all of them from the longest down, so that
    // short ones fill the end
    const int x = wg % kXcds, i = wg / kXcds, nbk = grid / (rowblocks * nsplit);
    int rank = 0;
    if (nbk >= kXcds) {
      const int mine = nbk / kXcds;
      w.bk = x * mine + i % mine;
      rank = i / mine;
    } else {
      const int per = kXcds / nbk;
      w.bk = x / per;
      rank = i * per + x % per;
    }
    w.rb = rowblocks - 1 - rank / nsplit;
    w.split = rank % nsplit;
  } else {
    if (xcd_remap) wg = (wg % kXcds) * (grid / kXcds) + wg / kXcds;
    w.rb = wg % rowblocks;
    if (longest_first) w.rb = rowblocks - 1 - w.rb;
    w.split = (wg / rowblocks) % nsplit;
    w.bk = wg / (rowblocks * nsplit);
  }
  return w;
}

}  // namespace kvq
