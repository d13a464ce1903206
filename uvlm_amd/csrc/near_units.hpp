// near_units.hpp -- how the near field's lists are cut into units (k_units_work, k_units_fill in
// near.hip).  Plain arithmetic, used on the device and checked on the host by
// tests/cpp/near_units_check.cpp.
//
// Each target leaf's list is worked off in one or more runs of entries of about equal work, so that
// a wave never walks a list far longer than the others' (a leaf next to much smaller ones, a probe
// tree with few leaves) while the chip is idle.  A leaf's work is its lane steps: the bodies of its
// list times its passes over its splits.  It is cut into ceil(work / limit) units, limit = the larger
// of LANE_STEPS_MIN and 1/UNITS_AIM of all leaves' work: below LANE_STEPS_MIN the staging and the
// prefix sums cost more than the pairs they serve (32 and 64 steps: 8k ring 72 and 77 us; 128: 100
// us).  More units shorten the last wave: 4M two rings (86k leaves) 10.0 ms with 4096, 9.9 with 8192,
// 9.6 with 16384.
#pragma once
#include <cstdint>

namespace uvlm {

constexpr int      LANE_STEPS_MIN = 64;
constexpr uint64_t UNITS_AIM      = 16384;

// The limit for `work` lane steps in all.  Rounded up: work / limit <= UNITS_AIM then, which
// units_bound and units_multi_bound take.
constexpr uint64_t units_limit(uint64_t work)
{
  const uint64_t lim = (work + UNITS_AIM - 1) / UNITS_AIM;
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
// <= sum (1 + work / limit), and a leaf cut into several has more work than the limit.
constexpr int64_t units_bound(int64_t nleaf) { return nleaf + (int64_t)UNITS_AIM; }
constexpr int64_t units_multi_bound(int64_t nleaf) { return nleaf < (int64_t)UNITS_AIM ? nleaf : (int64_t)UNITS_AIM; }

}  // namespace uvlm
