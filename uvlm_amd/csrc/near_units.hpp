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

// Lanes of a near-field workgroup: 64 for short lists of many small leaves, else 256.  256 lanes share a
// staged chunk between four waves and leave fewer of them idle on a leaf of 33..64 targets (one
// split of 64), but a list of a few hundred pairs does not fill them, and with few leaves a wavefront
// each leaves the chip idle.  `pairs` is the mean number of pairs a leaf: list entries times the mean
// leaf sizes of both trees.  P2P with 64 against 256 lanes (524,288 bodies, theta 0.5; us):
//   pairs       40    133    560   1053   2034   3992   4864   7091  10445  16685
//   mixed      400    474    436    307    515    365    372    519    390   1147
//             1408   1541    957    573    719    436    432    544    401   1032
//   FP64       673    800    756    659    831    772    778    755    973   1669
//             1871   2039   1343    945   1030    773    777    761    785   1453
// Mixed: 64 below NARROW_MIXED (two rings at 6482 pairs: 902 against 880).  FP64 holds twice the LDS a
// lane and gains less from the shorter chunk: 64 below NARROW_FP64 (two rings of 60,000 at 2047 pairs
// are level, a thin helix at 3337 loses 22%).  Below 8192 leaves 64 lanes leave the chip idle unless
// lists are shorter still: 64 below nleaf / 8 pairs (FP64: 2482 leaves of 264 pairs 29 against 34 us,
// 4630 of 560 pairs 29 against 47; 1951 of 468 pairs 46 against 35, 390 of 480 pairs 21 against 16).
constexpr double  NARROW_MIXED = 6000.0, NARROW_FP64 = 1500.0;
constexpr int64_t NARROW_LEAVES = 8192;
// lanes: 64 or 256 where the caller asks for them (64 lanes hold leaves of up to 64 targets), else 0
constexpr bool units_wide(int64_t nleaf, int64_t max_leaf, double pairs, double narrow, int lanes)
{
  if (max_leaf > 64) return true;
  if (lanes) return lanes != 64;
  return pairs >= (nleaf < NARROW_LEAVES ? (double)(nleaf / 8) : narrow);
}

}  // namespace uvlm
