// tree.hip -- octree build and dual-tree traversal on the device.
//
// Compiled with -ffp-contract=off: the octant tests, the child-centre recurrence and the
// multipole acceptance test must round exactly as the reference writes them, because the
// tree and the interaction lists are compared bit-exactly.
//
// Octree (semantics of src/tree.hpp:7-113):
//   1. bounds: fmin/fmax reduction, X0 = (max+min)/2, R0 = max half-extent * 1.00001 (tree.hpp:7-26)
//   2. a 63-bit key per body: the octant digits of the 21 levels below the root, each
//      digit (x>cx)+2(y>cy)+4(z>cz) against the FP64 centre recurrence
//      c_{l+1} = c_l + (R0/2^(l+1))*(+-1) (tree.hpp:57, 86-92)
//   3. radix sort of (key, index): stable, so equal keys keep the input order.  Only the top
//      digits the tree can use are sorted: the previous build's depth plus one level; a cell
//      that must split below them flags the build, which then sorts all 21 digits again
//   4. cells straight from the sorted keys, all levels at once (k_cells_count): a cell splits iff
//      NBODY > ncrit (tree.hpp:43), so the cells that begin at body i are those of the levels
//      from the first digit in which i differs from i - 1 (if the cell they share splits) down to
//      the first level that i does not share with body i + ncrit.  One scan over the bodies
//      numbers them in pre-order, the order by (BodyOffset, level)
//   5. cell numbering of the reference: root 0, child groups appended in DFS pre-order of
//      their parents (tree.hpp:81-96), i.e. ChildOffset(p) = 1 + sum of NCHILD over internal
//      cells before p in pre-order
//   6. inside a leaf the bodies keep their input order (the reference stops sorting at the
//      leaf): each leaf's input indices are ranked among themselves
// Traversal (semantics of src/traverse.hpp:32-85): breadth-first over (target, source)
// pairs with the reference's split rule and MAC; outputs are appended with one atomic per
// block and category, then put in CSR rows by target, ascending in the source.
#include <cstdlib>
#include <cstring>

#include "common.hpp"

#include <rocprim/rocprim.hpp>

#include <algorithm>

namespace uvlm {

namespace {

constexpr int BLK = 256;

inline int nblocks(int64_t n, int b = BLK) { return (int)std::max<int64_t>(1, (n + b - 1) / b); }

__global__ void k_bounds_partial(const double *__restrict__ x, const double *__restrict__ y,
                                 const double *__restrict__ z, int64_t N, double *part)
{
  __shared__ double s[6][BLK];
  double mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x; i < N; i += (int64_t)gridDim.x * BLK) {
    const double v[3] = {x[i], y[i], z[i]};
    for (int d = 0; d < 3; d++) {
      mn[d] = fmin(v[d], mn[d]);
      mx[d] = fmax(v[d], mx[d]);
    }
  }
  for (int d = 0; d < 3; d++) {
    s[d][threadIdx.x]     = mn[d];
    s[3 + d][threadIdx.x] = mx[d];
  }
  __syncthreads();
  for (int w = BLK / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int d = 0; d < 3; d++) {
        s[d][threadIdx.x]     = fmin(s[d][threadIdx.x + w], s[d][threadIdx.x]);
        s[3 + d][threadIdx.x] = fmax(s[3 + d][threadIdx.x + w], s[3 + d][threadIdx.x]);
      }
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int d = 0; d < 6; d++) part[blockIdx.x * 6 + d] = s[d][0];
}

// Totals of a build (32-bit): cells per level, leaves per level, error bits (0: deeper than the key holds;
// 1: a split needs a digit below the sorted ones).
enum { TOT_LEVEL = 0, TOT_LEAVES = 24, TOT_ERR = 47, TOT_COUNT = 48 };
static_assert(4 * TOT_COUNT <= 8 * N_COUNTERS, "build totals");

// X0 and R0 exactly as tree.hpp:19-25 computes them from Xmin/Xmax (one workgroup of BLK;
// min and max are exact in any order, so the parallel reduction gives the serial result).
__global__ __launch_bounds__(BLK) void k_bounds_final(const double *part, int nb, double *X0R0, uint32_t *tot)
{
  __shared__ double s[6][BLK];
  if (threadIdx.x < TOT_COUNT) tot[threadIdx.x] = 0;  // the build's totals
  double mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int b = threadIdx.x; b < nb; b += BLK)
    for (int d = 0; d < 3; d++) {
      mn[d] = fmin(part[b * 6 + d], mn[d]);
      mx[d] = fmax(part[b * 6 + 3 + d], mx[d]);
    }
  for (int d = 0; d < 3; d++) {
    s[d][threadIdx.x]     = mn[d];
    s[3 + d][threadIdx.x] = mx[d];
  }
  __syncthreads();
  for (int w = BLK / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int d = 0; d < 3; d++) {
        s[d][threadIdx.x]     = fmin(s[d][threadIdx.x + w], s[d][threadIdx.x]);
        s[3 + d][threadIdx.x] = fmax(s[3 + d][threadIdx.x + w], s[3 + d][threadIdx.x]);
      }
    __syncthreads();
  }
  if (threadIdx.x != 0) return;
  for (int d = 0; d < 3; d++) {
    mn[d] = s[d][0];
    mx[d] = s[3 + d][0];
  }
  double X0[3], R0 = 0;
  for (int d = 0; d < 3; d++) X0[d] = (mx[d] + mn[d]) / 2;
  for (int d = 0; d < 3; d++) {
    R0 = fmax(X0[d] - mn[d], R0);
    R0 = fmax(mx[d] - X0[d], R0);
  }
  R0 *= 1.00001;
  X0R0[0] = X0[0];
  X0R0[1] = X0[1];
  X0R0[2] = X0[2];
  X0R0[3] = R0;
}

__global__ void k_keys(const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z,
                       int64_t N, const double *__restrict__ X0R0, uint64_t *__restrict__ keys,
                       uint32_t *__restrict__ idx)
{
  const int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x;
  if (i >= N) return;
  const double xi = x[i], yi = y[i], zi = z[i];
  double       cx = X0R0[0], cy = X0R0[1], cz = X0R0[2];
  const double R0 = X0R0[3];
  uint64_t     key = 0;
  for (int l = 0; l < KEY_LEVELS; l++) {
    const int o = (xi > cx) + ((yi > cy) << 1) + ((zi > cz) << 2);
    key         = (key << 3) | (uint64_t)o;
    const double r = R0 / (double)(1LL << (l + 1));
    cx += r * (double)(((o & 1) >> 0) * 2 - 1);
    cy += r * (double)(((o & 2) >> 1) * 2 - 1);
    cz += r * (double)(((o & 4) >> 2) * 2 - 1);
  }
  keys[i] = key;
  idx[i]  = (uint32_t)i;
}

__device__ __forceinline__ int digit_at(uint64_t key, int l) { return (int)((key >> (3 * (KEY_LEVELS - 1 - l))) & 7); }

// Leading octant digits two keys share, at most dlim (the digits that are sorted).
__device__ __forceinline__ int common_digits(uint64_t a, uint64_t b, int dlim)
{
  const uint64_t x = a ^ b;  // bit 63 of a key is clear
  return min(dlim, x ? (__clzll((long long)x) - 1) / 3 : KEY_LEVELS);
}

__global__ void k_zero_u32(int64_t n, uint32_t *__restrict__ p)
{
  const int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x;
  if (i < n) p[i] = 0;
}

// info[i] = number of cells that begin at body i | level of the first << 8.  With s the digits i
// shares with i - 1 (-1 for the first body) and D those it shares with i + ncrit (-1 past the end):
// the cell of level s around i exists and splits, or nothing begins here; then the cells of levels
// s + 1 .. max(s, D) + 1 do, and all but the last split.  Found with a few loads near i, where a
// pass per level over the cells took a launch, a scan and a host read-back each, and 8 binary
// searches one after another per cell (8k ring: tree 0.42 ms).
constexpr int COUNT_BLOCKS = 1024;
__global__ __launch_bounds__(BLK) void k_cells_count(int64_t N, int64_t ncrit, int dlim,
                                                     const uint64_t *__restrict__ keys, uint32_t *__restrict__ info,
                                                     uint32_t *__restrict__ tot)
{
  __shared__ uint32_t loc[TOT_COUNT];
  if (threadIdx.x < TOT_COUNT) loc[threadIdx.x] = 0;
  __syncthreads();
  for (int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x; i < N; i += (int64_t)gridDim.x * BLK) {
    const uint64_t ki = keys[i];
    const int      s  = i > 0 ? common_digits(keys[i - 1], ki, dlim) : -1;
    const int      D  = i + ncrit < N ? common_digits(ki, keys[i + ncrit], dlim) : -1;
    if (D >= dlim) atomicOr(&loc[TOT_ERR], dlim < KEY_LEVELS ? 2u : 1u);
    uint32_t out = 0;
    if (s < dlim) {
      bool split = s < 0;  // the cell of level s around i - 1 and i holds more than ncrit bodies
      if (!split && i >= ncrit) split = common_digits(keys[i - ncrit], ki, dlim) >= s;
      if (!split) {
        int64_t lo = i >= ncrit ? i - ncrit + 1 : 0, hi = i - 1;  // its first body is here
        while (lo < hi) {
          const int64_t mid = (lo + hi) >> 1;
          if (common_digits(keys[mid], ki, dlim) >= s) hi = mid;
          else lo = mid + 1;
        }
        split = lo + ncrit < N && common_digits(keys[lo + ncrit], ki, dlim) >= s;
      }
      if (split) {
        const int last = max(s, min(D, dlim - 1)) + 1;
        out            = (uint32_t)(last - s) | (uint32_t)(s + 1) << 8;
        for (int l = s + 1; l <= last; l++) atomicAdd(&loc[TOT_LEVEL + l], 1u);
        atomicAdd(&loc[TOT_LEAVES + last], 1u);
      }
    }
    info[i] = out;
  }
  __syncthreads();
  if (threadIdx.x < TOT_COUNT && loc[threadIdx.x]) {
    if (threadIdx.x == TOT_ERR) atomicOr(&tot[TOT_ERR], loc[TOT_ERR]);
    else atomicAdd(&tot[threadIdx.x], loc[threadIdx.x]);
  }
}

struct CellCount {
  __device__ __host__ int32_t operator()(uint32_t info) const { return (int32_t)(info & 255); }
};
struct Popcount {
  __device__ __host__ int32_t operator()(uint32_t m) const { return __builtin_popcount(m); }
};

// The cells that begin at body i, in pre-order: first body, end, parent, level | octant << 8;
// and each cell's octant in its parent's mask of children.
__global__ void k_cells_write(int64_t N, int64_t ncrit, int dlim, const uint64_t *__restrict__ keys,
                              const uint32_t *__restrict__ info, const int32_t *__restrict__ scan,
                              int32_t *__restrict__ rb, int32_t *__restrict__ re, int32_t *__restrict__ rpar,
                              int32_t *__restrict__ rlvl, uint32_t *__restrict__ mask)
{
  const int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x;
  if (i >= N) return;
  const int n = info[i] & 255, l0 = info[i] >> 8;
  if (n == 0) return;
  const uint64_t ki = keys[i];
  const int      p0 = scan[i], last = l0 + n - 1;
  int            par = -1;
  if (i > 0) {  // the parent of the first cell begins at the first body that shares l0 - 1 digits
    int64_t lo = 0, hi = i - 1;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (common_digits(keys[mid], ki, dlim) >= l0 - 1) hi = mid;
      else lo = mid + 1;
    }
    par = scan[lo] + (l0 - 1 - (int)(info[lo] >> 8));
  }
  int64_t end = i + 1;
  for (int l = last; l >= l0; l--) {
    int64_t lo = end, hi = l == last ? min(N, i + ncrit) : N;  // first body that shares fewer than l digits
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (common_digits(keys[mid], ki, dlim) >= l) lo = mid + 1;
      else hi = mid;
    }
    end          = lo;
    const int p  = p0 + (l - l0), pp = l == l0 ? par : p - 1, o = l > 0 ? digit_at(ki, l - 1) : 0;
    rb[p]   = (int32_t)i;
    re[p]   = (int32_t)end;
    rpar[p] = pp;
    rlvl[p] = l | o << 8;
    if (pp >= 0) atomicOr(&mask[pp], 1u << o);
  }
}

// First slots of each level's cells and leaves.
struct LevelOffsets {
  int32_t off[KEY_LEVELS + 3], leaf[KEY_LEVELS + 3];
};

// Reference index of the cell with pre-order number p: 1 + children of the internal cells before
// its parent in pre-order + its siblings of lower octants.
__device__ __forceinline__ int cell_index(int p, const int32_t *rpar, const int32_t *rlvl, const int32_t *scan,
                                          const uint32_t *mask)
{
  const int q = rpar[p];
  return q < 0 ? 0 : 1 + scan[q] + __popc(mask[q] & ((1u << (rlvl[p] >> 8)) - 1u));
}

// The tree's arrays, from the cells in pre-order.  The centre is the recurrence of tree.hpp:86-92
// along the cell's digits.  Cells and leaves are listed by level, coarse first (the large leaves with the
// long lists start early), within a level in no fixed order (each block takes its range with one
// atomic per level): what walks them treats every cell by itself.
__global__ __launch_bounds__(BLK) void k_cells_out(
    int64_t C, LevelOffsets lo, const uint64_t *__restrict__ keys,
    const int32_t *__restrict__ rb, const int32_t *__restrict__ re, const int32_t *__restrict__ rpar,
    const int32_t *__restrict__ rlvl, const uint32_t *__restrict__ mask, const int32_t *__restrict__ scan,
    const double *__restrict__ X0R0, uint32_t *__restrict__ cursor, int32_t *__restrict__ c_nchild,
    int32_t *__restrict__ c_nbody, int32_t *__restrict__ c_child, int32_t *__restrict__ c_body,
    int32_t *__restrict__ c_level, int32_t *__restrict__ c_parent, double *__restrict__ cx, double *__restrict__ cy,
    double *__restrict__ cz, double *__restrict__ cR, int32_t *__restrict__ lvl_cells, int32_t *__restrict__ leaves)
{
  constexpr int       NL = KEY_LEVELS + 1;
  __shared__ uint32_t cnt[2 * NL], base[2 * NL];  // cells, then leaves
  if (threadIdx.x < 2 * NL) cnt[threadIdx.x] = 0;
  __syncthreads();
  const int64_t p = blockIdx.x * (int64_t)BLK + threadIdx.x;
  int           g = 0, l = 0;
  uint32_t      r = 0, rl = 0;
  bool          leaf = false;
  if (p < C) {
    l             = rlvl[p] & 255;
    g             = cell_index((int)p, rpar, rlvl, scan, mask);
    r             = atomicAdd(&cnt[l], 1u);
    const int nc  = __popc(mask[p]), b = rb[p];
    c_nchild[g]   = nc;
    c_nbody[g]    = re[p] - b;
    c_child[g]    = nc ? 1 + scan[p] : 0;
    c_body[g]     = b;
    c_level[g]    = l;
    c_parent[g]   = p == 0 ? -1 : cell_index(rpar[p], rpar, rlvl, scan, mask);
    const uint64_t key = keys[b];
    double         x = X0R0[0], y = X0R0[1], z = X0R0[2];
    const double   R0 = X0R0[3];
    for (int d = 0; d < l; d++) {
      const int    o = digit_at(key, d);
      const double h = R0 / (double)(1LL << (d + 1));
      x += h * (double)(((o & 1) >> 0) * 2 - 1);
      y += h * (double)(((o & 2) >> 1) * 2 - 1);
      z += h * (double)(((o & 4) >> 2) * 2 - 1);
    }
    cx[g] = x;
    cy[g] = y;
    cz[g] = z;
    cR[g] = R0 / (double)(1LL << l);
    leaf  = nc == 0;
    if (leaf) rl = atomicAdd(&cnt[NL + l], 1u);
  }
  __syncthreads();
  if (threadIdx.x < 2 * NL && cnt[threadIdx.x]) base[threadIdx.x] = atomicAdd(&cursor[threadIdx.x], cnt[threadIdx.x]);
  __syncthreads();
  if (p < C) lvl_cells[lo.off[l] + base[l] + r] = g;
  if (leaf) leaves[lo.leaf[l] + base[NL + l] + rl] = g;
}

// Final order of each leaf's bodies: their input indices ascending.  One wavefront per leaf ranks
// them against each other in LDS (ncrit <= RANK_MAX), in place of a radix sort of all N by leaf.
constexpr int64_t RANK_MAX = 1024;
__global__ __launch_bounds__(64) void k_leaf_rank(const int32_t *__restrict__ leaves, const int32_t *__restrict__ c_body,
                                                  const int32_t *__restrict__ c_nbody,
                                                  const uint32_t *__restrict__ idx, uint32_t *__restrict__ perm)
{
  extern __shared__ uint32_t v[];
  const int g = leaves[blockIdx.x], b = c_body[g], n = c_nbody[g], lane = threadIdx.x;
  for (int j = lane; j < n; j += 64) v[j] = idx[b + j];
  __syncthreads();
  for (int j = lane; j < n; j += 64) {
    const uint32_t m = v[j];
    int            r = 0;
#pragma unroll 4
    for (int k = 0; k < n; k++) r += v[k] < m;
    perm[b + r] = m;
  }
}

// lb[input index] = first body of its leaf (one wavefront per leaf; lanes stride over its bodies)
__global__ void k_leaf_begin(int64_t nleafrec, const int32_t *__restrict__ leaves, const int32_t *__restrict__ c_body,
                             const int32_t *__restrict__ c_nbody, const uint32_t *__restrict__ idx,
                             uint32_t *__restrict__ lb)
{
  const int64_t w    = (blockIdx.x * (int64_t)BLK + threadIdx.x) >> 6;
  const int     lane = threadIdx.x & 63;
  if (w >= nleafrec) return;
  const int g = leaves[w], b = c_body[g], n = c_nbody[g];
  for (int i = lane; i < n; i += 64) lb[idx[b + i]] = (uint32_t)b;
}

__global__ void k_iota_u32(int64_t N, uint32_t *__restrict__ v)
{
  const int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x;
  if (i < N) v[i] = (uint32_t)i;
}

// GATHER_FIELDS fields per grid row (blockIdx.y): the state moves with full memory parallelism
// and each permutation entry is read once per group of fields.  Two fields per row moved 37
// fields of 4M bodies in 0.45 ms (5.6 TB/s, a plain copy 5.8 TB/s), four in 0.54 ms.
constexpr int GATHER_FIELDS = 2;
__global__ void k_gather_fields(const double *__restrict__ src, double *__restrict__ dst, int64_t scap, int64_t dcap,
                                const int32_t *__restrict__ perm, int64_t N, int nfields)
{
  const int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x;
  if (i >= N) return;
  const int64_t j  = perm[i];
  const int     f0 = blockIdx.y * GATHER_FIELDS, f1 = min(nfields, f0 + GATHER_FIELDS);
  double        v[GATHER_FIELDS];
  for (int f = f0; f < f1; f++) v[f - f0] = src[f * scap + j];
  for (int f = f0; f < f1; f++) dst[f * dcap + i] = v[f - f0];
}

// The listed state fields and the bodies' original indices (the last grid row) in one launch.
struct FieldList {
  uint8_t f[N_FIELDS + 1];
  int     n;
};
__global__ void k_gather_state(const double *__restrict__ src, double *__restrict__ dst, int64_t cap,
                               const int32_t *__restrict__ perm, int64_t N, FieldList fl,
                               const int32_t *__restrict__ osrc, int32_t *__restrict__ odst)
{
  const int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x;
  if (i >= N) return;
  const int64_t j = perm[i];
  const int     k = blockIdx.y * GATHER_FIELDS;
  if (k >= fl.n) {
    odst[i] = osrc[j];
    return;
  }
  const int64_t f0 = fl.f[k], f1 = fl.f[min(k + 1, fl.n - 1)];  // an odd last field twice
  const double  a = src[f0 * cap + j], b = src[f1 * cap + j];
  dst[f0 * cap + i] = a;
  dst[f1 * cap + i] = b;
}
static_assert(GATHER_FIELDS == 2, "k_gather_state takes two fields a row");

// ------------------------------- traversal -------------------------------------
struct TreeView {
  const int32_t *nchild, *child, *nbody;
  const double  *cx, *cy, *cz, *R;
};

// Counters of a traversal (64-bit, sc.counters): list sizes so far, flags (TF_FRONT: the frontier's
// buffer overflowed; TF_LONG: a row longer than ROW_LONG), the largest frontier, the frontier sizes of
// steps k, k + 1, k + 2 (mod 4), and the rows longer than ROW_RANK.  The host adds TF_P2P and TF_M2L
// where a list's size passes its buffer; after an overflow the traversal starts again with larger ones.
enum { TC_P2P = 0, TC_M2L = 1, TC_FLAGS = 2, TC_MAXF = 3, TC_FRONT = 4, TC_LONG = 8, TC_COUNT = 9 };
static_assert(TC_COUNT <= UNIT_COUNTERS, "traversal counters");
enum { TF_FRONT = 1, TF_P2P = 2, TF_M2L = 4, TF_LONG = 8 };

// One breadth-first step over the frontier's pairs.  Lanes are (pair, child of the split side), 32
// pairs a round.  A block takes up to eight rounds before it reserves its output ranges, one atomic
// per class: the same-address atomics are the traversal's only serialisation (one reservation per 32
// pairs made it 3.8 times slower on the 4M tree).  The loads of all rounds are issued together, at
// clamped indices without branches; small frontiers spread over more blocks with fewer rounds.
// gap > 0 (near-field option, off in the reference): a pair is also near when its bodies can come
// closer than gap, |dX| < gap + sqrt(3) (Rt + Rs), tested on squares (rounds as the oracle does).
__global__ __launch_bounds__(BLK) void k_traverse(const int2 *__restrict__ ft, TreeView T, TreeView S, double theta,
                                                  double gap, int2 *__restrict__ nxt, int64_t cap_f,
                                                  uint2 *__restrict__ p2p, int64_t cap_p, uint2 *__restrict__ m2l,
                                                  int64_t cap_m, unsigned long long *__restrict__ cnt, int step)
{
  constexpr int                 ROUNDS = 8, PAIRS = BLK / 8;
  __shared__ unsigned           tot[BLK / 64][3];
  __shared__ unsigned long long base[3];
  const int                     tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, ch = tid & 7;
  int64_t                       nf = (int64_t)cnt[TC_FRONT + (step & 3)];
  if (blockIdx.x == 0 && tid == 0) {
    cnt[TC_FRONT + ((step + 2) & 3)] = 0;
    atomicMax(&cnt[TC_MAXF], (unsigned long long)nf);
    if (nf > cap_f) atomicOr(&cnt[TC_FLAGS], (unsigned long long)TF_FRONT);
  }
  if (nf > cap_f) nf = 0;  // the frontier was not stored whole
  const int64_t per = PAIRS * min((int64_t)ROUNDS, (nf + (int64_t)PAIRS * gridDim.x - 1) / ((int64_t)PAIRS * gridDim.x));
  for (int64_t b0 = blockIdx.x * per; b0 < nf; b0 += gridDim.x * per) {
    const int64_t b1 = min(nf, b0 + per);
    const int     nr = (int)((b1 - b0 + PAIRS - 1) / PAIRS);
    int           a[ROUNDS], b[ROUNDS], cls[ROUNDS];  // 0 push, 1 P2P, 2 M2L, 3 none
    auto          rounds = [&](auto count) {
      constexpr int R = decltype(count)::value;
      int           nct[R], ncs[R], fc[R];
      double        Rt[R], Rsrc[R];
#pragma unroll
      for (int r = 0; r < R; r++) {
        const int2 pr = ft[min(b0 + r * PAIRS + (tid >> 3), b1 - 1)];
        a[r] = pr.x, b[r] = pr.y;
      }
#pragma unroll
      for (int r = 0; r < R; r++) {
        nct[r] = T.nchild[a[r]], ncs[r] = S.nchild[b[r]];
        Rt[r] = T.R[a[r]], Rsrc[r] = S.R[b[r]];
        fc[r] = T.child[a[r]];
      }
#pragma unroll
      for (int r = 0; r < R; r++) {
        const bool split_t = ncs[r] == 0 || (Rt[r] >= Rsrc[r] && nct[r] != 0);
        const int  sc = S.child[b[r]];
        const bool on = ch < (split_t ? nct[r] : ncs[r]) && b0 + r * PAIRS + (tid >> 3) < b1;
        if (on && split_t) a[r] = fc[r] + ch;
        if (on && !split_t) b[r] = sc + ch;
        cls[r] = on ? 0 : 3;
      }
#pragma unroll
      for (int r = 0; r < R; r++) {
        const double dx = T.cx[a[r]] - S.cx[b[r]], dy = T.cy[a[r]] - S.cy[b[r]], dz = T.cz[a[r]] - S.cz[b[r]];
        const double D2 = dx * dx + dy * dy + dz * dz, R2 = D2 * theta * theta;
        const double Rs = T.R[a[r]] + S.R[b[r]];
        const double Gs = gap + 1.7320508075688772 * Rs;
        const int    k  = R2 < Rs * Rs || (gap > 0.0 && D2 < Gs * Gs)
                              ? (T.nchild[a[r]] == 0 && S.nchild[b[r]] == 0 ? 1 : 0)
                              : 2;
        if (cls[r] == 0) cls[r] = k;
      }
#pragma unroll
      for (int r = R; r < ROUNDS; r++) a[r] = b[r] = 0, cls[r] = 3;
    };
    if (nr <= 1) rounds(std::integral_constant<int, 1>{});
    else if (nr <= 2) rounds(std::integral_constant<int, 2>{});
    else if (nr <= 4) rounds(std::integral_constant<int, 4>{});
    else rounds(std::integral_constant<int, ROUNDS>{});
    unsigned sum[3] = {0, 0, 0};
#pragma unroll
    for (int r = 0; r < ROUNDS; r++)
      for (int k = 0; k < 3; k++) sum[k] += (unsigned)__popcll(__ballot(cls[r] == k));
    __syncthreads();  // the last pass's bases are read
    if (lane == 0)
      for (int k = 0; k < 3; k++) tot[wv][k] = sum[k];
    __syncthreads();
    if (tid < 3) {
      unsigned n = 0;
      for (int w = 0; w < BLK / 64; w++) n += tot[w][tid];
      const int slot = tid == 0 ? TC_FRONT + ((step + 1) & 3) : tid == 1 ? TC_P2P : TC_M2L;
      base[tid]      = n ? atomicAdd(&cnt[slot], (unsigned long long)n) : 0;
    }
    __syncthreads();
    int64_t at[3];
    for (int k = 0; k < 3; k++) {
      at[k] = (int64_t)base[k];
      for (int w = 0; w < wv; w++) at[k] += tot[w][k];
    }
    const unsigned long long below = (1ull << lane) - 1;
#pragma unroll
    for (int r = 0; r < ROUNDS; r++)
      for (int k = 0; k < 3; k++) {
        const unsigned long long m = __ballot(cls[r] == k);
        const int64_t            q = at[k] + __popcll(m & below);
        at[k] += __popcll(m);
        if (cls[r] != k) continue;
        if (k == 0) {
          if (q < cap_f) nxt[q] = make_int2(a[r], b[r]);
        } else if (k == 1) {
          if (q < cap_p) p2p[q] = make_uint2((unsigned)b[r], (unsigned)a[r]);
        } else if (q < cap_m) m2l[q] = make_uint2((unsigned)b[r], (unsigned)a[r]);
      }
  }
}

// The first `steps` (at most FIRST_STEPS) steps of a traversal in block 0, the frontier in LDS: the
// root pair (0, 0) is the first one, or, when both roots are leaves, the single P2P pair
// (traverse.hpp:41-44).  They hold 1, 8, 64 and 512 pairs at most, a launch each that cost 10 us
// mostly of launch and atomics (8192-body ring: 5 launches, 47 us with the gaps; here 15).  Clears the
// counters, the near-field units' too; the other blocks clear the nrows row counts.
constexpr int FIRST_STEPS = 4, FIRST_PAIRS = 512, FIRST_LANES = 1024;
static_assert(FIRST_PAIRS == 1 << 3 * (FIRST_STEPS - 1), "frontier of the last first step");
__global__ __launch_bounds__(FIRST_LANES) void k_traverse_first(TreeView T, TreeView S, double theta, double gap,
                                                                int steps, int2 *__restrict__ nxt, int64_t cap_f,
                                                                uint2 *__restrict__ p2p, int64_t cap_p,
                                                                uint2 *__restrict__ m2l, int64_t cap_m,
                                                                unsigned long long *__restrict__ cnt,
                                                                uint32_t *__restrict__ rows, int64_t nrows)
{
  const int tid = threadIdx.x;
  if (blockIdx.x > 0) {
    for (int64_t i = (blockIdx.x - 1) * (int64_t)FIRST_LANES + tid; i < nrows; i += (gridDim.x - 1) * (int64_t)FIRST_LANES)
      rows[i] = 0;
    return;
  }
  constexpr int       WAVES = FIRST_LANES / 64;
  __shared__ int2     fr[2][FIRST_PAIRS];
  __shared__ unsigned tot[WAVES][3];
  const int           lane = tid & 63, wv = tid >> 6, ch = tid & 7;
  const bool          leaves = T.nchild[0] == 0 && S.nchild[0] == 0;
  if (leaves && tid == 0) p2p[0] = make_uint2(0, 0);
  if (tid == 0) fr[0][0] = make_int2(0, 0);
  unsigned n = leaves ? 0 : 1, most = n;
  unsigned base[3] = {0, leaves ? 1u : 0u, 0};  // pushed, P2P, M2L so far
  __syncthreads();
  for (int st = 0; st < steps; st++) {
    const bool last = st == steps - 1;
    base[0]         = 0;
    for (unsigned b0 = 0; b0 < n; b0 += FIRST_LANES / 8) {
      const unsigned i = b0 + (tid >> 3);
      const int2     pr = fr[st & 1][min(i, n - 1)];
      int            a = pr.x, b = pr.y;
      const int      nct = T.nchild[a], ncs = S.nchild[b];
      const bool     split_t = ncs == 0 || (T.R[a] >= S.R[b] && nct != 0);
      const bool     on = ch < (split_t ? nct : ncs) && i < n;
      if (on && split_t) a = T.child[a] + ch;
      if (on && !split_t) b = S.child[b] + ch;
      int cls = 3;  // 0 push, 1 P2P, 2 M2L, 3 none (k_traverse)
      if (on) {
        const double dx = T.cx[a] - S.cx[b], dy = T.cy[a] - S.cy[b], dz = T.cz[a] - S.cz[b];
        const double D2 = dx * dx + dy * dy + dz * dz, R2 = D2 * theta * theta;
        const double Rs = T.R[a] + S.R[b];
        const double Gs = gap + 1.7320508075688772 * Rs;
        cls = R2 < Rs * Rs || (gap > 0.0 && D2 < Gs * Gs) ? (T.nchild[a] == 0 && S.nchild[b] == 0 ? 1 : 0) : 2;
      }
      unsigned long long m[3];
      for (int k = 0; k < 3; k++) m[k] = __ballot(cls == k);
      if (lane == 0)
        for (int k = 0; k < 3; k++) tot[wv][k] = (unsigned)__popcll(m[k]);
      __syncthreads();
      unsigned at[3];
      for (int k = 0; k < 3; k++) {
        at[k] = base[k] + (unsigned)__popcll(m[k] & ((1ull << lane) - 1));
        for (int w = 0; w < WAVES; w++) {
          if (w < wv) at[k] += tot[w][k];
          base[k] += tot[w][k];
        }
      }
      if (cls == 0) {
        if (!last) fr[(st + 1) & 1][at[0]] = make_int2(a, b);
        else if (at[0] < cap_f) nxt[at[0]] = make_int2(a, b);
      } else if (cls == 1) {
        if (at[1] < cap_p) p2p[at[1]] = make_uint2((unsigned)b, (unsigned)a);
      } else if (cls == 2 && at[2] < cap_m) m2l[at[2]] = make_uint2((unsigned)b, (unsigned)a);
      __syncthreads();
    }
    n    = base[0];
    most = max(most, n);
  }
  if (tid >= N_COUNTERS) return;
  unsigned long long v = 0;
  if (tid == TC_P2P) v = base[1];
  if (tid == TC_M2L) v = base[2];
  if (tid == TC_MAXF) v = most;
  if (tid == TC_FRONT + (steps & 3)) v = n;
  if (steps == 0 && tid == TC_FRONT && !leaves) {  // no step here: the root pair is the frontier
    nxt[0] = make_int2(0, 0);
    v      = 1;
  }
  cnt[tid] = v;
}

// ---- lists to CSR ---------------------------------------------------------------
// Pairs are (x = source, y = target), read as 64-bit keys target << 32 | source by the sort below.
// Rows of the CSR are filled by counting (each pair takes the next place of its row), then every row
// is put in ascending source order by one wavefront that ranks its entries against each other in
// LDS, or by a workgroup's bitonic sort from ROW_RANK entries on (ranking is quadratic).  Against two
// radix sorts of all pairs by (target, source), with their searches for the row starts: a quarter of
// the launches and half the time for small trees.  Large lists stay with the radix sort: the counting
// atomics go to the memory side (a row's entries lie on different XCDs), 23 a ns at best, and fall
// behind it from some million pairs on (100k rings, 0.39M pairs: lists phase 0.39 -> 0.26 ms; 60k cube
// with c = 6, 4.2M pairs in long rows: 0.55 ms sorted, 1.0 counted; 4M rings, 12.6M: 1.08 and 1.28).
// The size is that of the last lists built here; rows of more than ROW_LONG entries do not fit in
// LDS, and such lists are radix-sorted too.
constexpr int     ROW_RANK = 256, ROW_LONG = 16384;
constexpr int64_t ROWS_SORTED = 3 << 20;

// place[i] = number of pairs of the same row before pair i, in no fixed order; rows counts them.
// i < n0 are P2P pairs (rows 0..C), the others M2L pairs (rows C + 1 ..).
__global__ void k_row_count(int64_t C, unsigned long long *cnt, int64_t cap_p, int64_t cap_m,
                            const uint2 *__restrict__ p2p, const uint2 *__restrict__ m2l, uint32_t *__restrict__ rows,
                            uint32_t *__restrict__ place)
{
  const int64_t n0 = min((int64_t)cnt[TC_P2P], cap_p), n1 = min((int64_t)cnt[TC_M2L], cap_m);
  for (int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x; i < n0 + n1; i += (int64_t)gridDim.x * BLK) {
    const unsigned t = i < n0 ? p2p[i].y : m2l[i - n0].y;
    const uint32_t q = atomicAdd(&rows[(i < n0 ? 0 : C + 1) + t], 1u);
    place[i]         = q;
    if (q >= ROW_LONG) atomicOr(&cnt[TC_FLAGS], (unsigned long long)TF_LONG);
  }
}

// The same for few rows: a block counts its pairs in LDS and reserves each row's places at once.  The
// atomics on memory are then one a block and row, where every pair's atomic on a few hundred rows is
// serialised there (200003 bodies, 4096 probes: k_row_count 121 us, here 7; 8192-body ring, some
// thousand rows less contended: 11.4 and 7.1).  ROWS_LDS rows clear and flush in 8 steps a lane for
// the ROW_ITEMS pairs it counts; more rows would cost more than the pairs.
constexpr int ROWS_LDS = 2048, ROW_ITEMS = 8, ROW_CHUNK = BLK * ROW_ITEMS;
__global__ __launch_bounds__(BLK) void k_row_count_lds(int64_t C, unsigned long long *cnt, int64_t cap_p,
                                                       int64_t cap_m, const uint2 *__restrict__ p2p,
                                                       const uint2 *__restrict__ m2l, uint32_t *__restrict__ rows,
                                                       uint32_t *__restrict__ place)
{
  __shared__ uint32_t h[ROWS_LDS];
  const int64_t       n0 = min((int64_t)cnt[TC_P2P], cap_p), n1 = min((int64_t)cnt[TC_M2L], cap_m);
  const int           nr = (int)(2 * (C + 1));
  for (int64_t c0 = blockIdx.x * (int64_t)ROW_CHUNK; c0 < n0 + n1; c0 += gridDim.x * (int64_t)ROW_CHUNK) {
    for (int r = threadIdx.x; r < nr; r += BLK) h[r] = 0;
    __syncthreads();
    int      row[ROW_ITEMS];
    uint32_t q[ROW_ITEMS];
#pragma unroll
    for (int k = 0; k < ROW_ITEMS; k++) {
      const int64_t i = c0 + k * BLK + threadIdx.x;
      row[k]          = i < n0 ? (int)p2p[i].y : i < n0 + n1 ? (int)(C + 1 + m2l[i - n0].y) : -1;
    }
#pragma unroll
    for (int k = 0; k < ROW_ITEMS; k++) q[k] = row[k] >= 0 ? atomicAdd(&h[row[k]], 1u) : 0;
    __syncthreads();
    for (int r = threadIdx.x; r < nr; r += BLK) {
      const uint32_t n = h[r];
      if (n == 0) continue;
      const uint32_t at = atomicAdd(&rows[r], n);
      h[r]              = at;
      if (at + n > (uint32_t)ROW_LONG) atomicOr(&cnt[TC_FLAGS], (unsigned long long)TF_LONG);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < ROW_ITEMS; k++)
      if (row[k] >= 0) place[c0 + k * BLK + threadIdx.x] = h[row[k]] + q[k];
    __syncthreads();
  }
}

// Row starts of both lists (rowoff: the exclusive scan of the counts, P2P rows then M2L rows) and the
// pairs' sources at their places.
__global__ void k_row_fill(int64_t C, const unsigned long long *__restrict__ cnt, int64_t cap_p, int64_t cap_m,
                           const uint2 *__restrict__ p2p, const uint2 *__restrict__ m2l,
                           const uint32_t *__restrict__ rowoff, const uint32_t *__restrict__ place,
                           int32_t *__restrict__ off_p, int32_t *__restrict__ src_p, int32_t *__restrict__ off_m,
                           int32_t *__restrict__ src_m)
{
  const int64_t  n0 = min((int64_t)cnt[TC_P2P], cap_p), n1 = min((int64_t)cnt[TC_M2L], cap_m);
  const uint32_t m0 = rowoff[C + 1];
  for (int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x; i < max(n0 + n1, C + 1); i += (int64_t)gridDim.x * BLK) {
    if (i <= C) {
      off_p[i] = (int32_t)rowoff[i];
      off_m[i] = (int32_t)(rowoff[C + 1 + i] - m0);
    }
    if (i < n0) {
      const uint2 pr                     = p2p[i];
      src_p[rowoff[pr.y] + place[i]] = (int32_t)pr.x;
    } else if (i < n0 + n1) {
      const uint2 pr                              = m2l[i - n0];
      src_m[rowoff[C + 1 + pr.y] - m0 + place[i]] = (int32_t)pr.x;
    }
  }
}

// Every row of both lists in ascending order, one wavefront per row (rows r < C: P2P).
__global__ __launch_bounds__(BLK) void k_row_sort(int64_t C, const int32_t *__restrict__ off_p,
                                                  int32_t *__restrict__ src_p, const int32_t *__restrict__ off_m,
                                                  int32_t *__restrict__ src_m, unsigned long long *__restrict__ nlong,
                                                  uint32_t *__restrict__ longs)
{
  __shared__ __align__(16) int v[BLK / 64][ROW_RANK + 4];
  const int      wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t  r  = blockIdx.x * (int64_t)(BLK / 64) + wv;
  if (r >= 2 * C) return;
  const int32_t *off = r < C ? off_p + r : off_m + (r - C);
  int32_t       *src = (r < C ? src_p : src_m) + off[0];
  const int      n   = off[1] - off[0];
  if (n <= 1) return;
  if (n > ROW_RANK) {
    if (lane == 0) longs[atomicAdd(nlong, 1ull)] = (uint32_t)r;
    return;
  }
  int *w = v[wv];
  int  m[ROW_RANK / 64], q[ROW_RANK / 64];
#pragma unroll
  for (int i = 0; i < ROW_RANK / 64; i++) {
    const int j = lane + 64 * i;
    m[i]        = j < n ? src[j] : 0x7fffffff;
    q[i]        = 0;
    if (64 * i < n + 4) w[j] = m[i];
  }
  __builtin_amdgcn_wave_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  auto rank = [&](auto count) {
    for (int k = 0; k < n; k += 4) {  // entries past the end compare greater
      const int4 e = *reinterpret_cast<const int4 *>(w + k);
#pragma unroll
      for (int i = 0; i < decltype(count)::value; i++)
        q[i] += (e.x < m[i]) + (e.y < m[i]) + (e.z < m[i]) + (e.w < m[i]);
    }
  };
  if (n <= 64) rank(std::integral_constant<int, 1>{});
  else if (n <= 128) rank(std::integral_constant<int, 2>{});
  else rank(std::integral_constant<int, ROW_RANK / 64>{});
#pragma unroll
  for (int i = 0; i < ROW_RANK / 64; i++)
    if (lane + 64 * i < n) src[q[i]] = m[i];
}

// The rows k_row_sort left, a workgroup each.  A row holds a source cell once, so its order is a bit
// map of the Cs <= ROW_BITS source cells: set the entries' bits, count the bits below each word, write
// the set bits out.  Linear in the entries and in Cs / 32, where the bitonic sort takes log^2 steps with
// a barrier each (200003 bodies, 4096 probes, rows of thousands of entries: 80 us, here
// 7.3).
constexpr int BITS_LANES = 512, BITS_BLOCKS = 512, ROW_WORDS = 7168, ROW_BITS = 32 * ROW_WORDS;
__global__ __launch_bounds__(BITS_LANES) void k_row_sort_bits(int64_t C, int64_t Cs, const int32_t *__restrict__ off_p,
                                                              int32_t *__restrict__ src_p,
                                                              const int32_t *__restrict__ off_m,
                                                              int32_t *__restrict__ src_m,
                                                              const unsigned long long *__restrict__ nlong,
                                                              const uint32_t *__restrict__ longs)
{
  __shared__ unsigned bits[ROW_WORDS];
  __shared__ int      below[ROW_WORDS], ws[BITS_LANES / 64];
  const int           nl = (int)*nlong, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int           W = (int)((Cs + 31) / 32), per = (W + BITS_LANES - 1) / BITS_LANES;
  const int           w0 = min(W, tid * per), w1 = min(W, w0 + per);
  for (int k = blockIdx.x; k < nl; k += gridDim.x) {
    const int64_t  r   = longs[k];
    const int32_t *off = r < C ? off_p + r : off_m + (r - C);
    int32_t       *src = (r < C ? src_p : src_m) + off[0];
    const int      n   = off[1] - off[0];
    for (int w = tid; w < W; w += BITS_LANES) bits[w] = 0;
    __syncthreads();
    for (int j = tid; j < n; j += BITS_LANES) {
      const unsigned c = (unsigned)src[j];
      if (c < (unsigned)Cs) atomicOr(&bits[c >> 5], 1u << (c & 31));
    }
    __syncthreads();
    int sum = 0;
    for (int w = w0; w < w1; w++) {
      below[w] = sum;
      sum += __popc(bits[w]);
    }
    int inc = sum;
    for (int d = 1; d < 64; d *= 2) {
      const int v = __shfl_up(inc, d, 64);
      if (lane >= d) inc += v;
    }
    if (lane == 63) ws[wv] = inc;
    __syncthreads();
    int at = inc - sum;
    for (int v = 0; v < wv; v++) at += ws[v];
    for (int w = w0; w < w1; w++) below[w] += at;
    __syncthreads();
    for (int w = tid; w < W; w += BITS_LANES) {
      int q = below[w];
      for (unsigned b = bits[w]; b; b &= b - 1, q++)
        if (q < n) src[q] = 32 * w + __builtin_ctz(b);
    }
    __syncthreads();
  }
}

// The rows k_row_sort left, a workgroup each: bitonic sort of the next power of two entries, for
// source trees beyond k_row_sort_bits.
constexpr int LONG_LANES = 512, LONG_BLOCKS = 512;
__global__ __launch_bounds__(LONG_LANES) void k_row_sort_long(int64_t C, const int32_t *__restrict__ off_p,
                                                              int32_t *__restrict__ src_p,
                                                              const int32_t *__restrict__ off_m,
                                                              int32_t *__restrict__ src_m,
                                                              const unsigned long long *__restrict__ nlong,
                                                              const uint32_t *__restrict__ longs)
{
  __shared__ int v[ROW_LONG];
  const int      nl = (int)*nlong;
  for (int k = blockIdx.x; k < nl; k += gridDim.x) {
    const int64_t  r   = longs[k];
    const int32_t *off = r < C ? off_p + r : off_m + (r - C);
    int32_t       *src = (r < C ? src_p : src_m) + off[0];
    const int      n   = off[1] - off[0];
    if (n > ROW_LONG) continue;  // flagged: the radix sort takes the lists
    int m = 2 * ROW_RANK;
    while (m < n) m *= 2;
    for (int j = threadIdx.x; j < m; j += LONG_LANES) v[j] = j < n ? src[j] : 0x7fffffff;
    for (int w = 2; w <= m; w *= 2)
      for (int d = w / 2; d > 0; d /= 2) {
        __syncthreads();
        for (int j = threadIdx.x; j < m / 2; j += LONG_LANES) {
          const int  a = 2 * j - (j & (d - 1)), b = a + d;
          const bool up = (a & w) == 0;
          const int  x = v[a], y = v[b];
          if ((x > y) == up) v[a] = y, v[b] = x;
        }
      }
    __syncthreads();
    for (int j = threadIdx.x; j < n; j += LONG_LANES) src[j] = v[j];
    __syncthreads();
  }
}

// The pairs of the transposed lists (row = the source cell), one wavefront per row of both lists.
__global__ __launch_bounds__(BLK) void k_transpose_pairs(int64_t Ct, const int32_t *__restrict__ off_p,
                                                         const int32_t *__restrict__ src_p, int64_t n0,
                                                         const int32_t *__restrict__ off_m,
                                                         const int32_t *__restrict__ src_m,
                                                         uint2 *__restrict__ pairs_p, uint2 *__restrict__ pairs_m,
                                                         unsigned long long *__restrict__ cnt,
                                                         uint32_t *__restrict__ rows, int64_t nrows)
{
  for (int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x; i < nrows; i += gridDim.x * (int64_t)BLK) rows[i] = 0;
  const int64_t r = blockIdx.x * (int64_t)(BLK / 64) + (threadIdx.x >> 6);
  const int     lane = threadIdx.x & 63;
  if (r == 0 && lane < N_COUNTERS)
    cnt[lane] = lane == TC_P2P ? (unsigned long long)n0 : lane == TC_M2L ? (unsigned long long)off_m[Ct] : 0;
  if (r >= 2 * Ct) return;
  const bool     near = r < Ct;
  const int64_t  t    = near ? r : r - Ct;
  const int32_t *off  = near ? off_p : off_m, *src = near ? src_p : src_m;
  uint2         *out  = near ? pairs_p : pairs_m;
  for (int q = off[t] + lane; q < off[t + 1]; q += 64) out[q] = make_uint2((unsigned)t, (unsigned)src[q]);
}

// Keys (row << lbits) | entry of the radix sort.
__global__ void k_pack_keys(int64_t n, const uint2 *__restrict__ pairs, int lbits, uint64_t *__restrict__ keys)
{
  const int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x;
  if (i < n) keys[i] = (uint64_t)pairs[i].y << lbits | pairs[i].x;
}

// List keys are (row << lbits) | entry, sorted: off[c] = the first key of row c.
__global__ void k_csr(int64_t C, const uint64_t *__restrict__ keys, int64_t n, int lbits, int32_t *__restrict__ off)
{
  const int64_t c = blockIdx.x * (int64_t)BLK + threadIdx.x;
  if (c > C) return;
  const uint64_t want = (uint64_t)c << lbits;
  int64_t        lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (keys[mid] < want) lo = mid + 1;
    else hi = mid;
  }
  off[c] = (int32_t)lo;
}

__global__ void k_low_bits(int64_t n, const uint64_t *__restrict__ keys, int lbits, int32_t *__restrict__ out)
{
  const int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x;
  if (i < n) out[i] = (int32_t)(uint32_t)(keys[i] & ((1ull << lbits) - 1));
}

void h2d(hipStream_t s, void *d, const void *h, size_t bytes)
{
  UVLM_HIP(hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, s));
  UVLM_HIP(hipStreamSynchronize(s));
}

// The host waits for n values at d.  A kernel writes them to the handle's page-locked words: a copy to
// pageable memory is staged and waited for by the runtime, some 25 us more each (a step of 600 bodies,
// two such waits: 407 -> 345 us; 8192-body ring 902 -> 845).
__global__ __launch_bounds__(64) void k_to_host(int n, const uint32_t *__restrict__ d, uint32_t *__restrict__ h)
{
  for (int i = threadIdx.x; i < n; i += 64) h[i] = d[i];
}

template <class T> void to_host(hipStream_t s, Scratch &sc, T *h, const void *d, size_t n = 1)
{
  static_assert(sizeof(T) % 4 == 0, "words");
  if (!sc.back.h || sizeof(T) * n > HostWords::BYTES) {
    UVLM_HIP(hipMemcpyAsync(h, d, sizeof(T) * n, hipMemcpyDeviceToHost, s));
    UVLM_HIP(hipStreamSynchronize(s));
    return;
  }
  k_to_host<<<1, 64, 0, s>>>((int)(sizeof(T) * n / 4), (const uint32_t *)d, sc.back.d);
  UVLM_LAUNCH_CHECK();
  UVLM_HIP(hipStreamSynchronize(s));
  std::memcpy(h, sc.back.h, sizeof(T) * n);
}

void sort_keys_u64(hipStream_t s, Scratch &sc, uint64_t *in, uint64_t *out, int64_t n, int end_bit)
{
  size_t bytes = 0;
  UVLM_HIP(rocprim::radix_sort_keys(nullptr, bytes, in, out, (size_t)n, 0, end_bit, s));
  sc.sort_tmp.reserve(bytes);
  UVLM_HIP(rocprim::radix_sort_keys(sc.sort_tmp.p, bytes, in, out, (size_t)n, 0, end_bit, s));
}

template <class In, class T> void excl_scan(hipStream_t s, Scratch &sc, In in, T *out, int64_t n)
{
  size_t bytes = 0;
  UVLM_HIP(rocprim::exclusive_scan(nullptr, bytes, in, out, T(0), (size_t)n, rocprim::plus<T>(), s));
  sc.scan_tmp.reserve(bytes);
  UVLM_HIP(rocprim::exclusive_scan(sc.scan_tmp.p, bytes, in, out, T(0), (size_t)n, rocprim::plus<T>(), s));
}

int bits_for(int64_t v)
{
  int b = 1;
  while (b < 63 && (int64_t(1) << b) <= v) b++;
  return b;
}

}  // namespace

// ---------------------------------------------------------------------------------
void build_tree(hipStream_t s, Scratch &sc, const double *x, const double *y, const double *z, int64_t N,
                int64_t ncrit, Tree &tree, int32_t *perm_out)
{
  if (N <= 0) throw Error(UVLM_ERR_ARG, "empty particle set");
  if (N >= (int64_t(1) << 31)) throw Error(UVLM_ERR_ARG, "more than 2^31-1 particles");
  // 1. bounds
  const int nb = std::min(1024, nblocks(N));
  sc.partial.reserve(sizeof(double) * 6 * nb);
  tree.X0R0.reserve(sizeof(double) * 4);
  k_bounds_partial<<<nb, BLK, 0, s>>>(x, y, z, N, sc.partial.as<double>());
  sc.counters.reserve(8 * N_COUNTERS);
  uint32_t *tot = sc.counters.as<uint32_t>();
  k_bounds_final<<<1, BLK, 0, s>>>(sc.partial.as<double>(), nb, tree.X0R0.as<double>(), tot);
  UVLM_LAUNCH_CHECK();
  // 2-3. keys and stable sort
  sc.keys0.reserve(8 * N);
  sc.keys1.reserve(8 * N);
  sc.idx0.reserve(4 * N);
  sc.idx1.reserve(4 * N);
  const uint64_t *keys = sc.keys1.as<uint64_t>();
  const uint32_t *idx  = sc.idx1.as<uint32_t>();
  uint32_t       *info = sc.idx0.as<uint32_t>();  // free once sorted
  int32_t        *scan = sc.keys0.as<int32_t>();
  int            dlim = std::min(KEY_LEVELS, std::max(1, tree.sort_digits));
  uint32_t  h[TOT_COUNT];
  for (;;) {
    k_keys<<<nblocks(N), BLK, 0, s>>>(x, y, z, N, tree.X0R0.as<double>(), sc.keys0.as<uint64_t>(),
                                       sc.idx0.as<uint32_t>());
    UVLM_LAUNCH_CHECK();
    // stable sort of (key, index) on the top dlim digits
    size_t    bytes = 0;
    const int b0    = 3 * (KEY_LEVELS - dlim);
    UVLM_HIP(rocprim::radix_sort_pairs(nullptr, bytes, sc.keys0.as<uint64_t>(), sc.keys1.as<uint64_t>(),
                                       sc.idx0.as<uint32_t>(), sc.idx1.as<uint32_t>(), (size_t)N, b0, 3 * KEY_LEVELS,
                                       s));
    sc.sort_tmp.reserve(bytes);
    UVLM_HIP(rocprim::radix_sort_pairs(sc.sort_tmp.p, bytes, sc.keys0.as<uint64_t>(), sc.keys1.as<uint64_t>(),
                                       sc.idx0.as<uint32_t>(), sc.idx1.as<uint32_t>(), (size_t)N, b0, 3 * KEY_LEVELS,
                                       s));
    // 4. cells, numbered in pre-order
    k_cells_count<<<std::min(COUNT_BLOCKS, nblocks(N)), BLK, 0, s>>>(N, ncrit, dlim, keys, info, tot);
    UVLM_LAUNCH_CHECK();
    excl_scan(s, sc, rocprim::make_transform_iterator(info, CellCount{}), scan, N);
    to_host(s, sc, h, tot, TOT_COUNT);
    if (h[TOT_ERR] & 1) throw Error(UVLM_ERR_DEPTH, "more than ncrit coincident bodies: octree deeper than 21 levels");
    if (!(h[TOT_ERR] & 2)) break;
    dlim = KEY_LEVELS;  // a cell splits below the sorted digits: all of them, again from the keys
    k_zero_u32<<<1, BLK, 0, s>>>(TOT_COUNT, tot);
  }
  LevelOffsets         lo{};
  std::vector<int64_t> off{0};
  int64_t              nleaf = 0;
  for (int l = 0; l <= KEY_LEVELS && h[TOT_LEVEL + l]; l++) {
    lo.off[l]  = (int32_t)off.back();
    lo.leaf[l] = (int32_t)nleaf;
    off.push_back(off.back() + h[TOT_LEVEL + l]);
    nleaf += h[TOT_LEAVES + l];
  }
  const int64_t C    = off.back();
  const int     nlev = (int)off.size() - 1;
  tree.sort_digits   = nlev;  // digits 0 .. nlev-1: this tree's splits plus one spare level
  tree.C             = C;
  tree.nlevels       = nlev;
  tree.nleaf         = nleaf;
  tree.lvl_off       = off;

  // 5. numbering
  for (DevBuf *b : {&sc.rec_begin, &sc.rec_end, &sc.rec_parent, &sc.rec_level, &sc.rec_scan}) b->reserve(4 * C);
  sc.rec_mask.reserve(4 * (C + TOT_COUNT));
  for (DevBuf *b : {&tree.nchild, &tree.nbody, &tree.child, &tree.body, &tree.level, &tree.parent, &tree.lvl_cells})
    b->reserve(4 * C);
  for (DevBuf *b : {&tree.cx, &tree.cy, &tree.cz, &tree.R}) b->reserve(8 * C);
  tree.leaves.reserve(4 * tree.nleaf);
  int32_t  *rb = sc.rec_begin.as<int32_t>(), *re = sc.rec_end.as<int32_t>(), *rpar = sc.rec_parent.as<int32_t>();
  int32_t  *rlvl = sc.rec_level.as<int32_t>(), *cscan = sc.rec_scan.as<int32_t>();
  uint32_t *mask = sc.rec_mask.as<uint32_t>(), *cursor = mask + C;
  k_zero_u32<<<nblocks(C + TOT_COUNT), BLK, 0, s>>>(C + TOT_COUNT, mask);
  k_cells_write<<<nblocks(N), BLK, 0, s>>>(N, ncrit, dlim, keys, info, scan, rb, re, rpar, rlvl, mask);
  UVLM_LAUNCH_CHECK();
  excl_scan(s, sc, rocprim::make_transform_iterator(mask, Popcount{}), cscan, C);
  k_cells_out<<<nblocks(C), BLK, 0, s>>>(
      C, lo, keys, rb, re, rpar, rlvl, mask, cscan, tree.X0R0.as<double>(), cursor, tree.nchild.as<int32_t>(),
      tree.nbody.as<int32_t>(), tree.child.as<int32_t>(), tree.body.as<int32_t>(), tree.level.as<int32_t>(),
      tree.parent.as<int32_t>(), tree.cx.as<double>(), tree.cy.as<double>(), tree.cz.as<double>(),
      tree.R.as<double>(), tree.lvl_cells.as<int32_t>(), tree.leaves.as<int32_t>());
  UVLM_LAUNCH_CHECK();

  // 6. final permutation
  if (ncrit <= RANK_MAX) {
    k_leaf_rank<<<(int)tree.nleaf, 64, 4 * ncrit, s>>>(tree.leaves.as<int32_t>(), tree.body.as<int32_t>(),
                                                       tree.nbody.as<int32_t>(), idx, (uint32_t *)perm_out);
    UVLM_LAUNCH_CHECK();
    return;
  }
  // large leaves: the input indices 0..N-1, stably sorted by their leaf's first body
  uint32_t *lb = sc.keys0.as<uint32_t>(), *lb_sorted = sc.keys1.as<uint32_t>(), *iota = sc.idx0.as<uint32_t>();
  k_leaf_begin<<<nblocks(tree.nleaf * 64), BLK, 0, s>>>(tree.nleaf, tree.leaves.as<int32_t>(),
                                                        tree.body.as<int32_t>(), tree.nbody.as<int32_t>(), idx, lb);
  k_iota_u32<<<nblocks(N), BLK, 0, s>>>(N, iota);
  UVLM_LAUNCH_CHECK();
  {
    size_t bytes = 0;
    UVLM_HIP(rocprim::radix_sort_pairs(nullptr, bytes, lb, lb_sorted, iota, (uint32_t *)perm_out, (size_t)N, 0,
                                       bits_for(N), s));
    sc.sort_tmp.reserve(bytes);
    UVLM_HIP(rocprim::radix_sort_pairs(sc.sort_tmp.p, bytes, lb, lb_sorted, iota, (uint32_t *)perm_out, (size_t)N, 0,
                                       bits_for(N), s));
  }
}

void gather_fields(hipStream_t s, const double *src, double *dst, int64_t src_cap, int64_t dst_cap, int nfields,
                   const int32_t *perm, int64_t N)
{
  if (N <= 0 || nfields <= 0) return;
  k_gather_fields<<<dim3(nblocks(N), (nfields + GATHER_FIELDS - 1) / GATHER_FIELDS), BLK, 0, s>>>(
      src, dst, src_cap, dst_cap, perm, N, nfields);
  UVLM_LAUNCH_CHECK();
}

void gather_state(hipStream_t s, const double *src, double *dst, int64_t cap, const uint8_t *fields, int nfields,
                  const int32_t *osrc, int32_t *odst, const int32_t *perm, int64_t N)
{
  if (N <= 0) return;
  FieldList fl{};
  fl.n = nfields;
  for (int k = 0; k < nfields; k++) fl.f[k] = fields[k];
  k_gather_state<<<dim3(nblocks(N), (nfields + GATHER_FIELDS - 1) / GATHER_FIELDS + 1), BLK, 0, s>>>(
      src, dst, cap, perm, N, fl, osrc, odst);
  UVLM_LAUNCH_CHECK();
}

// Largest value of x[0..n) (non-negative values): per-block maxima, then one block over them.
__global__ void k_max_partial(const double *__restrict__ x, int64_t n, double *__restrict__ part)
{
  __shared__ double red[BLK];
  double            m = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLK) m = fmax(m, x[i]);
  red[threadIdx.x] = m;
  __syncthreads();
  for (int o = BLK / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + o]);
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

double max_value(hipStream_t s, Scratch &sc, const double *x, int64_t n)
{
  if (n <= 0) return 0.0;
  const int nb = (int)std::min<int64_t>(512, (n + BLK - 1) / BLK);
  sc.partial.reserve(sizeof(double) * (nb + 1));
  double *part = sc.partial.as<double>();
  k_max_partial<<<nb, BLK, 0, s>>>(x, n, part);
  k_max_partial<<<1, BLK, 0, s>>>(part, nb, part + nb);
  UVLM_LAUNCH_CHECK();
  double m = 0.0;
  to_host(s, sc, &m, part + nb);
  return m;
}

static TreeView view(const Tree &t)
{
  return TreeView{(const int32_t *)t.nchild.p, (const int32_t *)t.child.p, (const int32_t *)t.nbody.p,
                  (const double *)t.cx.p,      (const double *)t.cy.p,      (const double *)t.cz.p,
                  (const double *)t.R.p};
}

// CSR rows by target of the np P2P and nm M2L pairs in sc.out_p2p / out_m2l (their numbers are read
// on the device; np and nm bound them).  C target cells, Cs source cells; zeroed: the caller has
// cleared the row counts.
static void rows_by_counting(hipStream_t s, Scratch &sc, int64_t C, int64_t Cs, int64_t np, int64_t nm, bool zeroed,
                             Lists &l)
{
  unsigned long long *cnt = sc.counters.as<unsigned long long>();
  l.p2p_off.reserve(4 * (C + 1));
  l.m2l_off.reserve(4 * (C + 1));
  l.p2p_src.reserve(4 * std::max<int64_t>(np, 1));
  l.m2l_src.reserve(4 * std::max<int64_t>(nm, 1));
  sc.row_cnt.reserve(4 * 2 * (C + 1));
  sc.row_off.reserve(4 * 2 * (C + 1));
  sc.row_place.reserve(4 * std::max<int64_t>(np + nm, 1));
  sc.row_long.reserve(4 * ((np + nm) / ROW_RANK + 1));
  uint32_t    *rows = sc.row_cnt.as<uint32_t>(), *ro = sc.row_off.as<uint32_t>(), *pl = sc.row_place.as<uint32_t>();
  const uint2 *p2p = sc.out_p2p.as<uint2>(), *m2l = sc.out_m2l.as<uint2>();
  const int    grid = (int)std::min<int64_t>(4096, nblocks(std::max<int64_t>(np + nm, C + 1)));
  if (!zeroed) k_zero_u32<<<nblocks(2 * (C + 1)), BLK, 0, s>>>(2 * (C + 1), rows);
  if (2 * (C + 1) <= ROWS_LDS)
    k_row_count_lds<<<(int)std::min<int64_t>(4096, (np + nm) / ROW_CHUNK + 1), BLK, 0, s>>>(
        C, cnt, np, nm, p2p, m2l, rows, pl);
  else k_row_count<<<grid, BLK, 0, s>>>(C, cnt, np, nm, p2p, m2l, rows, pl);
  excl_scan(s, sc, rows, ro, 2 * (C + 1));
  k_row_fill<<<grid, BLK, 0, s>>>(C, cnt, np, nm, p2p, m2l, ro, pl, l.p2p_off.as<int32_t>(), l.p2p_src.as<int32_t>(),
                                  l.m2l_off.as<int32_t>(), l.m2l_src.as<int32_t>());
  k_row_sort<<<nblocks(2 * C, BLK / 64), BLK, 0, s>>>(C, l.p2p_off.as<int32_t>(), l.p2p_src.as<int32_t>(),
                                                      l.m2l_off.as<int32_t>(), l.m2l_src.as<int32_t>(),
                                                      cnt + TC_LONG, sc.row_long.as<uint32_t>());
  const bool may_long = np + nm > ROW_RANK && Cs > ROW_RANK;  // a row holds a source cell once
  if (may_long && Cs <= ROW_BITS)
    k_row_sort_bits<<<BITS_BLOCKS, BITS_LANES, 0, s>>>(C, Cs, l.p2p_off.as<int32_t>(), l.p2p_src.as<int32_t>(),
                                                       l.m2l_off.as<int32_t>(), l.m2l_src.as<int32_t>(), cnt + TC_LONG,
                                                       sc.row_long.as<uint32_t>());
  else if (may_long)
    k_row_sort_long<<<LONG_BLOCKS, LONG_LANES, 0, s>>>(C, l.p2p_off.as<int32_t>(), l.p2p_src.as<int32_t>(),
                                                       l.m2l_off.as<int32_t>(), l.m2l_src.as<int32_t>(), cnt + TC_LONG,
                                                       sc.row_long.as<uint32_t>());
  UVLM_LAUNCH_CHECK();
}

// The same by a radix sort of the pairs (rows of any length); the sizes are known here.
static void rows_by_sorting(hipStream_t s, Scratch &sc, int64_t C, int64_t Cs, Lists &l)
{
  const int lbits = bits_for(std::max<int64_t>(Cs, 1)), eb = lbits + bits_for(std::max<int64_t>(C, 1));
  for (int which = 0; which < 2; which++) {
    const int64_t n   = which == 0 ? l.np2p : l.nm2l;
    DevBuf       &raw = which == 0 ? sc.out_p2p : sc.out_m2l;
    DevBuf       &off = which == 0 ? l.p2p_off : l.m2l_off;
    DevBuf       &src = which == 0 ? l.p2p_src : l.m2l_src;
    off.reserve(4 * (C + 1));
    src.reserve(4 * std::max<int64_t>(n, 1));
    sc.keys0.reserve(8 * std::max<int64_t>(n, 1));
    sc.keys1.reserve(8 * std::max<int64_t>(n, 1));
    if (n > 0) {
      k_pack_keys<<<nblocks(n), BLK, 0, s>>>(n, raw.as<uint2>(), lbits, sc.keys0.as<uint64_t>());
      sort_keys_u64(s, sc, sc.keys0.as<uint64_t>(), sc.keys1.as<uint64_t>(), n, eb);
    }
    k_csr<<<nblocks(C + 1), BLK, 0, s>>>(C, sc.keys1.as<uint64_t>(), n, lbits, off.as<int32_t>());
    k_low_bits<<<nblocks(n), BLK, 0, s>>>(n, sc.keys1.as<uint64_t>(), lbits, src.as<int32_t>());
    UVLM_LAUNCH_CHECK();
  }
}

// The near-field units as read back into cnt, made again with fewer rows of partial sums while there is no
// room for them.
static void take_units(hipStream_t s, Scratch &sc, const Tree &tt, const Tree &st, int64_t max_leaf,
                       unsigned long long *cnt, Lists &l)
{
  unsigned long long *dcnt = sc.counters.as<unsigned long long>();
  while (!near_units_set(sc, cnt + UNIT_COUNTERS, l)) {
    near_units_enqueue(s, sc, tt, st, max_leaf, dcnt + TC_P2P, false, l, (uint64_t)l.n_rows / 8);
    to_host(s, sc, cnt, dcnt, N_COUNTERS);
  }
}

// max_leaf >= 0: also the lists' near-field units (near.hip), read back together with the sizes.
void traverse(hipStream_t s, Scratch &sc, const Tree &tt, const Tree &st, double theta, Lists &lists, double gap,
              int64_t max_leaf)
{
  TreeView T = view(tt), S = view(st);
  int64_t cap_f = std::max<int64_t>(4096, 8 * (tt.C + st.C));
  int64_t cap_p = std::max<int64_t>(4096, 32 * tt.nleaf);
  int64_t cap_m = std::max<int64_t>(4096, 64 * tt.C);
  if (const char *e = std::getenv("UVLM_LIST_CAPACITY")) {  // first sizes of fresh buffers (tests of the regrowth)
    const long long v = std::atoll(e);
    if (v > 0) cap_f = cap_p = cap_m = v;
  }
  sc.front0.reserve(8 * cap_f);
  sc.front1.reserve(8 * cap_f);
  sc.out_p2p.reserve(8 * cap_p);
  sc.out_m2l.reserve(8 * cap_m);
  sc.counters.reserve(8 * N_COUNTERS);
  unsigned long long *dcnt = sc.counters.as<unsigned long long>();
  // every step splits one side of each pair, so a frontier of two trees of known depth is empty after
  // their levels' sum; trees handed in by a caller are walked until it is
  const int  depth = tt.nlevels > 0 && st.nlevels > 0 ? tt.nlevels + st.nlevels - 2 : -1;
  constexpr int BATCH = 6;
  for (;;) {
    cap_f = std::min(sc.front0.bytes, sc.front1.bytes) / 8;
    cap_p = sc.out_p2p.bytes / 8;
    cap_m = sc.out_m2l.bytes / 8;
    unsigned long long cnt[N_COUNTERS] = {};
    // with lists of this kind built before, their size picks the way and the sizes are read back with
    // the units; without, the sizes are read first
    // trees handed in by a caller are always sorted: cells there may share children, and ranking a
    // row takes its sources to be distinct
    const bool    own   = depth >= 0;
    const bool    ahead = own && lists.np2p > 0 && !lists.long_rows && lists.np2p + lists.nm2l <= ROWS_SORTED;
    const int     first = own ? std::min(depth, FIRST_STEPS) : FIRST_STEPS;
    const int64_t nrows = ahead || (own && lists.np2p == 0) ? 2 * (tt.C + 1) : 0;  // counts that may be needed
    if (nrows) sc.row_cnt.reserve(4 * nrows);
    k_traverse_first<<<1 + (int)std::min<int64_t>(256, (nrows + 4 * FIRST_LANES - 1) / (4 * FIRST_LANES)), FIRST_LANES, 0,
                       s>>>(T, S, theta, gap, first, (first & 1 ? sc.front1 : sc.front0).as<int2>(), cap_f,
                            sc.out_p2p.as<uint2>(), cap_p, sc.out_m2l.as<uint2>(), cap_m, dcnt,
                            sc.row_cnt.as<uint32_t>(), nrows);
    UVLM_LAUNCH_CHECK();
    int64_t most = std::min<int64_t>((int64_t)1 << 3 * first, cap_f);  // pairs a step's frontier can hold
    for (int k = first;; k++) {
      if (depth >= 0 ? k >= depth : k > first && (k - first) % BATCH == 0) {
        if (depth >= 0) break;
        to_host(s, sc, cnt, dcnt, TC_COUNT);
        if (cnt[TC_FRONT + (k & 3)] == 0 || (cnt[TC_FLAGS] & TF_FRONT)) break;
      }
      DevBuf &fin = k & 1 ? sc.front1 : sc.front0, &fout = k & 1 ? sc.front0 : sc.front1;
      k_traverse<<<(int)std::min<int64_t>(2048, nblocks(most, BLK / 8)), BLK, 0, s>>>(
          fin.as<int2>(), T, S, theta, gap, fout.as<int2>(), cap_f, sc.out_p2p.as<uint2>(), cap_p,
          sc.out_m2l.as<uint2>(), cap_m, dcnt, k);
      UVLM_LAUNCH_CHECK();
      most = std::min<int64_t>(8 * most, cap_f);
    }
    bool units_clear = true;  // the units' counters (k_traverse_first)
    auto units       = [&] {
      if (max_leaf >= 0) near_units_enqueue(s, sc, tt, st, max_leaf, dcnt + TC_P2P, units_clear, lists);
      units_clear = false;
    };
    auto by_counting = [&](int64_t np, int64_t nm) {
      rows_by_counting(s, sc, tt.C, st.C, np, nm, nrows > 0, lists);
      units();
    };
    if (ahead) by_counting(cap_p, cap_m);
    to_host(s, sc, cnt, dcnt, N_COUNTERS);
    if (depth >= 0 && !(cnt[TC_FLAGS] & TF_FRONT) && cnt[TC_FRONT + (depth & 3)] != 0)
      throw Error(UVLM_ERR_INTERNAL, "the traversal did not end");
    int over = (int)(cnt[TC_FLAGS] & TF_FRONT);
    if ((int64_t)cnt[TC_P2P] > cap_p) over |= TF_P2P;
    if ((int64_t)cnt[TC_M2L] > cap_m) over |= TF_M2L;
    if (over) {  // grow what overflowed (at least doubled) and traverse again
      if (over & TF_FRONT) {
        const int64_t want = std::max<int64_t>(2 * cap_f, 2 * (int64_t)cnt[TC_MAXF]);
        sc.front0.reserve(8 * want);
        sc.front1.reserve(8 * want);
      }
      if (over & TF_P2P) sc.out_p2p.reserve(8 * std::max<int64_t>(2 * cap_p, 2 * (int64_t)cnt[TC_P2P]));
      if (over & TF_M2L) sc.out_m2l.reserve(8 * std::max<int64_t>(2 * cap_m, 2 * (int64_t)cnt[TC_M2L]));
      continue;
    }
    lists.np2p = (int64_t)cnt[TC_P2P];
    lists.nm2l = (int64_t)cnt[TC_M2L];
    if (own && !ahead && !lists.long_rows && lists.np2p + lists.nm2l <= ROWS_SORTED) {
      by_counting(lists.np2p, lists.nm2l);
      to_host(s, sc, cnt, dcnt, N_COUNTERS);
    } else if (!ahead) cnt[TC_FLAGS] |= TF_LONG;
    if (cnt[TC_FLAGS] & TF_LONG) {
      lists.long_rows = lists.long_rows || lists.np2p + lists.nm2l <= ROWS_SORTED;
      rows_by_sorting(s, sc, tt.C, st.C, lists);
      units();
      if (max_leaf >= 0) to_host(s, sc, cnt, dcnt, N_COUNTERS);
    }
    if (max_leaf >= 0) take_units(s, sc, tt, st, max_leaf, cnt, lists);
    return;
  }
}

void transpose_lists(hipStream_t s, Scratch &sc, const Tree &in_targets, const Tree &in_sources, const Lists &in,
                     Lists &out, int64_t max_leaf)
{
  const int64_t Ct = in_targets.C, Cs = in_sources.C;
  out.np2p = in.np2p;
  out.nm2l = in.nm2l;
  sc.out_p2p.reserve(8 * std::max<int64_t>(in.np2p, 1));
  sc.out_m2l.reserve(8 * std::max<int64_t>(in.nm2l, 1));
  sc.counters.reserve(8 * N_COUNTERS);
  unsigned long long *dcnt   = sc.counters.as<unsigned long long>();
  const bool          sorted = out.long_rows || in.np2p + in.nm2l > ROWS_SORTED;
  const int64_t       nrows  = sorted ? 0 : 2 * (Cs + 1);
  if (nrows) sc.row_cnt.reserve(4 * nrows);
  k_transpose_pairs<<<nblocks(2 * Ct, BLK / 64), BLK, 0, s>>>(
      Ct, in.p2p_off.as<int32_t>(), in.p2p_src.as<int32_t>(), in.np2p, in.m2l_off.as<int32_t>(),
      in.m2l_src.as<int32_t>(), sc.out_p2p.as<uint2>(), sc.out_m2l.as<uint2>(), dcnt, sc.row_cnt.as<uint32_t>(), nrows);
  UVLM_LAUNCH_CHECK();
  unsigned long long cnt[N_COUNTERS] = {};
  if (!sorted) {
    rows_by_counting(s, sc, Cs, Ct, in.np2p, in.nm2l, true, out);
    near_units_enqueue(s, sc, in_sources, in_targets, max_leaf, dcnt + TC_P2P, true, out);
    to_host(s, sc, cnt, dcnt, N_COUNTERS);
    out.long_rows = (cnt[TC_FLAGS] & TF_LONG) != 0;
  }
  if (sorted || out.long_rows) {
    rows_by_sorting(s, sc, Cs, Ct, out);
    near_units_enqueue(s, sc, in_sources, in_targets, max_leaf, dcnt + TC_P2P, sorted, out);
    to_host(s, sc, cnt, dcnt, N_COUNTERS);
  }
  take_units(s, sc, in_sources, in_targets, max_leaf, cnt, out);
}

}  // namespace uvlm
