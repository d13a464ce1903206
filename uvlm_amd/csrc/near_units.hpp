// near_units.hpp -- how the near field's lists are cut into units (k_units_work, k_units_fill in
// near.hip).  Plain arithmetic, used on the device and checked on the host by
// tests/cpp/near_units_check.cpp.
//
// Each target leaf's list is worked off in one or more runs of entries of about equal work, so that
// a wave never walks a list far longer than the others' (a leaf next to much smaller ones, a probe
// tree with few leaves) while the chip is idle.  A leaf's work is its lane steps: the bodies of its
// list times its passes over its splits.  It is cut into ceil(work / limit) units, limit = the largest
// of LANE_STEPS_MIN, 1/UNITS_AIM of all leaves' work and what keeps the partial sums small: below LANE_STEPS_MIN the staging and the
// prefix sums cost more than the pairs they serve (32 and 64 steps: 8k ring 72 and 77 us; 128: 100
// us).  More units shorten the last wave: 4M two rings (86k leaves) 10.0 ms with 4096, 9.9 with 8192,
// 9.6 with 16384.
#pragma once
#include <cstdint>

namespace uvlm {

constexpr int      LANE_STEPS_MIN = 64;
constexpr uint64_t UNITS_AIM      = 16384;

// Rows of partial sums (12 doubles, one row a target of each unit of a leaf cut into several) at most:
// 6.4 GB.  Leaves of some hundred targets come nowhere near it (4M two rings, leaves of up to 192:
// 0.78M rows), leaves of thousands do (1M two rings, ncrit 4000: 25M).  Fewer, longer units cost such
// leaves time (with 4M rows at most: ncrit 1000 21.8 -> 24.3 ms, ncrit 4000 66 -> 88).
constexpr uint64_t UNITS_ROWS_MAX = 1 << 26;

// The limit for `work` lane steps in all, the sum `rowwork` of every leaf's targets times its lane steps,
// and at most `rows` rows.  Rounded up: work / limit <= UNITS_AIM and 2 rowwork / limit <= rows
// then, which the bounds below take.  rows = 0: every leaf is one unit.
constexpr uint64_t units_limit(uint64_t work, uint64_t rowwork, uint64_t rows)
{
  if (rows < 2) return UINT64_MAX / 2;
  const uint64_t a = (work + UNITS_AIM - 1) / UNITS_AIM, r = rowwork / (rows / 2) + 1;
  const uint64_t lim = a > r ? a : r;
  return lim > LANE_STEPS_MIN ? lim : LANE_STEPS_MIN;
}

// Units of a leaf with a list of len entries and `work` lane steps: at least one, at most one an entry.
constexpr int units_of_leaf(uint32_t work, int len, uint64_t lim)
{
  const uint64_t n = (work + lim - 1) / lim, most = len > 1 ? len : 1;
  return n < 1 ? 1 : (int)(n < most ? n : most);
}

// First entry of unit j of n over a list of len entries (j = n: its end).
constexpr int units_first(int len, int j, int n) { return (int)((int64_t)len * j / n); }

// Bounds of the units and of the leaves cut into several, over nleaf leaves: sum ceil(work / limit)
// <= sum (1 + work / limit), and a leaf cut into several has more work than the limit.  For the same
// reason its rows are at most 2 work / limit times its targets, `rows` over all leaves.
constexpr int64_t units_bound(int64_t nleaf) { return nleaf + (int64_t)UNITS_AIM; }
constexpr int64_t units_multi_bound(int64_t nleaf) { return nleaf < (int64_t)UNITS_AIM ? nleaf : (int64_t)UNITS_AIM; }

}  // namespace uvlm
