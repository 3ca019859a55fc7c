// Every (pair, row block, split) of a prefill launch is served by exactly one workgroup, for all launches
// that the host plans can make (tests/test_prefill_plan.py compiles and runs this).

#include <cstdio>
#include <vector>

#include "../myinfer_amd/csrc/prefill_plan.h"

using namespace kvq;

static long checked = 0;

static bool covers(const PrePlan& pl, const char* what, int a, int b, int c, int d) {
  const int grid = pl.nunits * pl.nsplit;
  const int xcd_remap = (int64_t)pl.nunits * pl.nsplit % kXcds == 0;  // as prefill_params sets it
  std::vector<char> seen(grid, 0);
  ++checked;
  for (int wg = 0; wg < grid; ++wg) {
    const PreWg w = prefill_wg(wg, grid, pl.rowblocks, pl.nsplit, xcd_remap, pl.longest_first);
    const bool in = w.bk >= 0 && w.bk < pl.nbk && w.rb >= 0 && w.rb < pl.rowblocks && w.split >= 0 && w.split < pl.nsplit;
    char* s = in ? &seen[((size_t)w.bk * pl.rowblocks + w.rb) * pl.nsplit + w.split] : nullptr;
    if (!s || *s) {
      std::printf("%s (%d %d %d %d): workgroup %d of %d serves pair %d/%d, row block %d/%d, split %d/%d%s, numbering %d\n", what,
                  a, b, c, d, wg, grid, w.bk, pl.nbk, w.rb, pl.rowblocks, w.split, pl.nsplit, s ? " again" : "",
                  pl.longest_first);
      return false;
    }
    *s = 1;
  }
  return true;  // grid workgroups, each a combination of its own: all of them
}

int main() {
  // every number of pairs, row blocks and splits
  for (int nbk = 1; nbk <= 16; ++nbk)
    for (int rowblocks = 1; rowblocks <= 128; ++rowblocks)
      for (int unequal = 0; unequal < 2; ++unequal)
        for (int ns = 1; ns <= 8; ++ns) {
          PrePlan pl{};
          pl.nbk = nbk;
          pl.rowblocks = rowblocks;
          pl.nunits = nbk * rowblocks;
          pl.tiles = 64;
          pl.unequal = unequal;
          set_splits(&pl, ns);
          if (!covers(pl, "pairs, row blocks, splits, unequal", nbk, rowblocks, ns, unequal)) return 1;
        }
  // the plans of prompts and chunks, with every smaller count of splits too (masked calls may run with one)
  const int heads[][3] = {{32, 4, 1}, {8, 1, 2}, {8, 1, 4}, {16, 4, 1}, {8, 2, 1}, {14, 2, 1}, {5, 1, 4}, {12, 4, 1},
                          {16, 2, 2}, {32, 8, 1}, {32, 32, 1}, {4, 4, 3}, {2, 1, 1}};
  for (const auto& h : heads)
    for (int L = 31; L <= 4100; L += 23)
      for (int S : {L, L + 777})
        for (int window : {0, 300})
          for (int causal : {0, 1}) {
            PrePlan pl = prefill_plan(h[2], h[0], h[1], L, S, window, causal);
            for (int ns = pl.nsplit; ns >= 1; --ns) {
              set_splits(&pl, ns);
              if (!covers(pl, "Hq, Hkv, B, L", h[0], h[1], h[2], L)) return 1;
            }
          }
  std::printf("%ld launches\n", checked);
  return 0;
}
