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

// How workgroups are numbered (prefill_wg).
enum PreOrder : int {
  kEqual,   // row blocks of about equal length
  kCausal,  // a causal prompt, whose first row blocks see few keys
  kMasked,  // a general mask, whose row blocks see what it says
};

struct PrePlan {
  int nbk, rowblocks, nunits, nsplit, tiles, chunk, order;
  int rep, lo;  // query heads of a KV head; keys before the call's first position
};

// Splits merged by the last of them to arrive; more take prefill_combine_kernel. Few splits are cheaper
// in the kernel (the last 512-token chunk of 16384, 4 splits: 155.2 against 161.3 us for the layer
// step), many in a launch of their own, whose loads run side by side: 64 rows of 4 KV heads over 8192
// keys (32 splits) 45.5 -> 18.4 us, over 32768 (64 splits) 81.2 -> 28.0.
constexpr int kPFusedMaxSplit = 4;

// The first row block with keys in split `split` of a causal prompt: its last row, at position lo + row /
// rep, sees key split * chunk. (Split 0 of every row block is run: it writes the rows that see no key.)
template <typename P>
constexpr int prefill_first_block(const P& p, int split) {
  if (p.order != kCausal || split == 0) return 0;
  const int64_t x = (int64_t)split * p.chunk - p.lo;
  return x <= 0 ? 0 : (int)std::min<int64_t>(p.rowblocks, x * p.rep / kPRows);
}

// The keys the rows [fr0, frl] of a row block see, in whole tiles ([lo, hi), lo rounded down to a
// tile), and the splits they are cut into: `chunk` keys each, so that workgroups of long and short
// row blocks (a causal prompt's last and first) are about as long, the short ones taking fewer.
struct KeySplit {
  int lo, hi, chunk, nsplit;
};
template <typename P>
constexpr KeySplit split_keys(const P& p, int S_b, int fr0, int frl) {
  const int pos_min = S_b - p.L + fr0 / p.rep, pos_max = S_b - p.L + frl / p.rep;
  KeySplit k{};
  k.hi = p.causal ? std::min(S_b, pos_max + 1) : S_b;
  k.lo = (p.window > 0 ? std::max(0, pos_min - p.window + 1) : 0) & ~(kPT - 1);
  const int span = std::max(k.hi - k.lo, 0);
  k.chunk = std::max(p.chunk, ((span + p.nsplit - 1) / p.nsplit + kPT - 1) / kPT * kPT);
  k.nsplit = std::max((span + k.chunk - 1) / k.chunk, 1);
  return k;
}

// Workgroups of a launch.
template <typename P>
constexpr int prefill_grid(const P& p) {
  int n = 0;
  for (int s = 0; s < p.nsplit; ++s) n += p.rowblocks - prefill_first_block(p, s);
  return p.nbk * n;
}

// Cut `pl` into `nsplit` splits. The chunk follows from the count here and nowhere else, so that every plan is
// numbered for the count it runs with.
inline void set_splits(PrePlan* pl, int nsplit) {
  pl->nsplit = nsplit;
  pl->chunk = (pl->tiles + nsplit - 1) / nsplit * kPT;
}

inline PrePlan prefill_plan(int B, int Hq, int Hkv, int L, int S, int window, int causal) {
  PrePlan pl;
  const int rep = Hq / Hkv, nrows = rep * L;
  pl.nbk = B * Hkv;
  pl.rowblocks = (nrows + kPRows - 1) / kPRows;
  pl.nunits = pl.nbk * pl.rowblocks;
  pl.rep = rep;
  pl.lo = S - L;
  // keys a row block sees: the whole context, or about a window; the first row block of a causal call
  const int span = window > 0 ? std::min(S, window + kPRows) : S;
  const int first = causal && window == 0 ? std::min(S, S - L + (kPRows + rep - 1) / rep) : span;
  const int tiles = (span + kPT - 1) / kPT, tiles0 = (first + kPT - 1) / kPT;
  pl.tiles = tiles;
  pl.order = 2 * tiles0 <= tiles ? kCausal : kEqual;
  int ns = (kPTargetWgs + pl.nunits - 1) / pl.nunits;
  if (pl.order == kCausal) {
    // The number of splits with the shortest estimate, in tiles (of about 1.75 us at 128 dims). The longest
    // workgroup's tiles and what it costs besides, merge included: 4 for one split, 7.5 to 8.5 for 2 to 4;
    // past them a merge launch, which grows with the row blocks and pays only where all workgroups run at
    // once. Where they do not, an even share of all the work (partials contend: a split more, 1.5 tiles more
    // for each) and a quarter of a workgroup, the last ones'.
    // In us, 8 bits, for 1 / 2 / 3 / 4 / 8 splits, 128 dims, heads and tokens:
    //   8 / 1 of 4096: 112 / 68 / 55 / 75 / -;  2 / 2 of 4096: 112 / 65 / 50 / 43 / 35;
    //   32 / 8 of 2048: 64 / 54 / 57 / 61 / -;  8 / 2 of 1500: 47 / 32 / 27 / 26 / 30.
    const float avg = 0.5f * (tiles + tiles0);
    float best = 0.0f;
    for (int c = 1; c <= kMaxSplit && (c <= kPFusedMaxSplit || pl.nunits * c <= kPTargetWgs); ++c) {
      if (c > 1 && 4 * c > tiles) break;
      set_splits(&pl, c);
      const int n = prefill_grid(pl);
      const float longest = pl.chunk / kPT + (c == 1 ? 4.0f : c <= kPFusedMaxSplit ? 6.5f + 0.5f * c : 7.0f + pl.nunits / 9.0f);
      const float share = (pl.nunits * avg + n * (c > 1 ? 3.5f + 1.5f * c : 4.0f)) / kPTargetWgs;
      const float est = n <= kPTargetWgs ? longest : std::max(longest, share + 0.25f * longest);
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

// Workgroup `wg` of the launch's `grid`: its (sequence, KV head) pair, row block and split, each combination
// that holds keys once.
struct PreWg {
  int bk, rb, split;
};
template <typename P>
constexpr PreWg prefill_wg(const P& p, int wg, int grid) {
  PreWg w{};
  if (p.order == kEqual) {
    // The row blocks of one (pair, split) share every K/V tile, so they are consecutive, and consecutive
    // workgroups are placed on one XCD (the hardware hands workgroups to the 8 XCDs in turn): each tile is
    // fetched into one L2 rather than eight.
    if (grid % kXcds == 0) wg = (wg % kXcds) * (grid / kXcds) + wg / kXcds;
    w.rb = wg % p.rowblocks;
    w.split = (wg / p.rowblocks) % p.nsplit;
    w.bk = wg / (p.rowblocks * p.nsplit);
  } else {
    // Row blocks of unequal length: pairs in turn (so that 8 or more stay on an XCD each), a split's row
    // blocks from the longest down, split 0, which has the short ones, last. Neighbours are of about
    // one length, so every XCD and shader engine, which take workgroups in turn, gets its share; and the
    // splits past a row block's keys have no workgroups, which would hold others up until they left.
    // (Splits in turn instead, all of them: an XCD gets one split's workgroups only where 8 or 4 divides
    // their number. 32 heads / 4 KV heads of 2000 tokens 75 -> 55 us, 8 / 1 of 4096 82 -> 55.)
    w.bk = wg % p.nbk;
    int rank = wg / p.nbk;
    w.split = p.nsplit - 1;
    for (; w.split > 0; --w.split) {
      const int n = p.rowblocks - prefill_first_block(p, w.split);
      if (rank < n) break;
      rank -= n;
    }
    w.rb = p.rowblocks - 1 - rank;
  }
  return w;
}

}  // namespace kvq
