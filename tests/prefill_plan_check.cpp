// The workgroups of a prefill launch (tests/test_prefill_plan.py compiles and runs this), for all launches that the
// host plans can make: every (pair, row block, split) that holds keys is served by exactly one, and so is split
// 0 of every row block; and the 8 XCDs, which take workgroups in turn, get equal shares of a causal prompt.

#include <cstdio>
#include <vector>

#include "../myinfer_amd/csrc/prefill_plan.h"

using namespace kvq;

static long checked = 0;

struct Call : PrePlan {  // a plan with what else the kernel reads
  int L, S, causal, window;
};

static bool covers(const Call& c, const char* what, int Hq, int Hkv, int B) {
  const int grid = prefill_grid(c), nrows = c.rep * c.L;
  std::vector<char> seen((size_t)c.nunits * c.nsplit, 0);
  double tiles[kXcds] = {0}, all = 0;
  ++checked;
  auto keys = [&](int rb, int split, int S_b) {
    const KeySplit k = split_keys(c, S_b, rb * kPRows, std::min((rb + 1) * kPRows, nrows) - 1);
    return split >= k.nsplit ? 0 : std::max(0, std::min(k.chunk, k.hi - k.lo - split * k.chunk));
  };
  for (int wg = 0; wg < grid; ++wg) {
    const PreWg w = prefill_wg(c, wg, grid);
    const bool in = w.bk >= 0 && w.bk < c.nbk && w.rb >= 0 && w.rb < c.rowblocks && w.split >= 0 && w.split < c.nsplit;
    char* s = in ? &seen[((size_t)w.bk * c.rowblocks + w.rb) * c.nsplit + w.split] : nullptr;
    if (!s || *s) {
      std::printf("%s %d/%d heads, B %d, L %d, S %d, window %d: workgroup %d of %d serves pair %d/%d, row block %d/%d, split %d/%d%s\n",
                  what, Hq, Hkv, B, c.L, c.S, c.window, wg, grid, w.bk, c.nbk, w.rb, c.rowblocks, w.split, c.nsplit,
                  s ? " again" : "");
      return false;
    }
    *s = 1;
    const double t = keys(w.rb, w.split, c.S) / (double)kPT + 4;  // (a workgroup costs some 4 tiles besides its own)
    tiles[wg % kXcds] += t;
    all += t;
  }
  for (int u = 0; u < c.nunits; ++u)
    for (int s = 0; s < c.nsplit; ++s) {
      if (seen[(size_t)u * c.nsplit + s]) continue;
      bool needed = s == 0 || c.order != kCausal;
      for (int S_b : {c.S, c.S - 1, c.S - 63, c.S - 200, c.L, c.S / 2}) needed |= keys(u % c.rowblocks, s, std::min(std::max(S_b, 0), c.S)) > 0;
      if (needed) {
        std::printf("%s %d/%d heads, B %d, L %d, S %d, window %d: row block %d/%d, split %d/%d is not served\n", what, Hq, Hkv, B,
                    c.L, c.S, c.window, u % c.rowblocks, c.rowblocks, s, c.nsplit);
        return false;
      }
    }
  if (c.order == kCausal && grid > 256 && (c.nbk % kXcds == 0 || c.nbk < kXcds))
    for (double t : tiles)
      if (t > 1.15 * all / kXcds) {
        std::printf("%s %d/%d heads, B %d, L %d, S %d, %d splits: an XCD gets %.0f tiles of %.0f\n", what, Hq, Hkv, B, c.L, c.S,
                    c.nsplit, t, all);
        return false;
      }
  return true;
}

int main() {
  // prompts and chunks, at their plan's number of splits, all smaller ones (masked calls may run with one) and
  // some larger
  const int heads[][3] = {{32, 4, 1}, {8, 1, 2}, {8, 1, 4}, {16, 4, 1}, {8, 2, 1}, {14, 2, 1}, {5, 1, 4}, {12, 4, 1},
                          {16, 2, 2}, {32, 8, 1}, {32, 32, 1}, {4, 4, 3}, {2, 1, 1}, {1, 1, 1}, {3, 3, 1}};
  for (const auto& h : heads)
    for (int L = 31; L <= 4100; L += 23)
      for (int S : {L, L + 777, L - 30})
        for (int window : {0, 300})
          for (int causal : {0, 1}) {
            Call c{prefill_plan(h[2], h[0], h[1], L, S, window, causal), L, S, causal, window};
            if (c.nsplit > 1 && c.order == kCausal && c.nunits * c.nsplit > 256 && c.nsplit > kPFusedMaxSplit) return 2;
            for (int ns = std::max(c.nsplit, 8); ns >= 1; --ns) {
              set_splits(&c, ns);
              if (!covers(c, "prompt", h[0], h[1], h[2])) return 1;
            }
            if (!causal && !window) {
              c.order = kMasked;
              for (int ns : {1, 3}) {
                set_splits(&c, ns);
                if (!covers(c, "masked", h[0], h[1], h[2])) return 1;
              }
            }
          }
  std::printf("%ld launches\n", checked);
  return 0;
}
