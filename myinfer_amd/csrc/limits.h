// Limits that the host plans and the kernels share.
#pragma once

#include <stddef.h>

namespace kvq {

constexpr int kXcds = 8;  // MI355X: 8 XCDs, each with its own L2
constexpr int kMaxSplit = 128;

// Launches whose last-arriving workgroup merges the splits count arrivals per unit in a counter
// block at the start of the workspace. Every launch reserves the same block, so launches of
// different shapes that share one workspace never place partials over another launch's counters;
// a launch with more units than this does not split (prefill) or merges with combine_kernel
// (decode). Counters start at zero (the workspace is zero-filled once) and the merging workgroup
// resets its own.
constexpr int kMaxCountedUnits = 65536;
constexpr size_t kCounterBytes = (size_t)kMaxCountedUnits * sizeof(unsigned);

}  // namespace kvq
