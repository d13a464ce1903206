// near.hip -- near-field P2P: regularised Biot-Savart velocity and velocity gradient.
//
// Kernel of src/multipoleKernels.hpp:223-301 (sensor form 303-341): for target i and
// source j with dX = x_i - x_j, R^2 != 0, s = R / (sqrt(2) sigma_j):
//   g  = erf(s) - (2/sqrt(pi)) s e^{-s^2},  f1 = g / (4 pi R^3),
//   f2 = (2 s^2 t2 - 3 g) / (4 pi R^5)      (t2 = (2/sqrt(pi)) s e^{-s^2})
//   u -= f1 (dX x a_j),   J[a][b] -= f2 (dX x a_j)_a dX_b + f1 eps_{abk} a_j,k.
// Only the source core size sigma_j enters (multipoleKernels.hpp:243).
//
// Layout: one workgroup of BLK lanes (64 or 256) per unit of a target leaf's list (near_units.hpp).
// Lanes = (target t) x (source split s): a pass takes ntp of the leaf's targets
// (near_targets_per_pass) and S = BLK / ntp splits, each taking every S-th source, and the partial
// sums are combined in a fixed order (LDS, no atomics).  The bodies of all source leaves in the
// unit's list entries are streamed through LDS in full chunks across leaf boundaries (prefix sums
// of the leaf sizes in LDS, binary search per slot), so small leaves do not pay a barrier per leaf.
//
// FP64 path: G = g/s^3 and its derivative in double (pair_kernel.hpp), two sources per step.
// Mixed path: FP32 arithmetic on coordinates relative to the target leaf centre (the source
// offsets are formed in FP64 while staging), two sources per step over zero-padded chunks (one
// trip count for all lanes), per-chunk FP32 partial sums added into FP64 per-target
// accumulators; G = g/s^3 and its derivative from pair_kernel.hpp.
#include "common.hpp"
#include "pair_kernel.hpp"

#include <algorithm>

namespace uvlm {

namespace {

// acc[0..2] += f1 c, acc[3..10] += f2 c (x) dX with c = dX x a, and acc[12..14] += f1 a: the
// f1 eps_{abk} a_k part of J is antisymmetric, so its sum is kept as one vector and folded
// into J once per chunk (fold_antisym) instead of six multiply-adds per pair.  c is
// perpendicular to dX, so c (x) dX is traceless and its zz entry (acc[11]) is formed from the
// xx and yy sums in fold_antisym.
__device__ __forceinline__ float  fma_(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fma_(double a, double b, double c) { return fma(a, b, c); }
template <class T>
__device__ __forceinline__ void accumulate_pair(T *acc, T dx, T dy, T dz, T ax, T ay, T az, T f1, T f2, bool withJ)
{
  const T cx = dy * az - dz * ay, cy = dz * ax - dx * az, cz = dx * ay - dy * ax;
  acc[0] = fma_(f1, cx, acc[0]);
  acc[1] = fma_(f1, cy, acc[1]);
  acc[2] = fma_(f1, cz, acc[2]);
  if (withJ) {
    const T k0 = f2 * cx, k1 = f2 * cy, k2 = f2 * cz;
    acc[3]  = fma_(k0, dx, acc[3]);
    acc[4]  = fma_(k0, dy, acc[4]);
    acc[5]  = fma_(k0, dz, acc[5]);
    acc[6]  = fma_(k1, dx, acc[6]);
    acc[7]  = fma_(k1, dy, acc[7]);
    acc[8]  = fma_(k1, dz, acc[8]);
    acc[9]  = fma_(k2, dx, acc[9]);
    acc[10] = fma_(k2, dy, acc[10]);
    acc[12] = fma_(f1, ax, acc[12]);
    acc[13] = fma_(f1, ay, acc[13]);
    acc[14] = fma_(f1, az, acc[14]);
  }
}
// J[2][2] = -(J[0][0] + J[1][1]) and J[a][b] += eps_{abk} F_k with F = acc[12..14] (row-major J
// in acc[3..11]).
template <class T> __device__ __forceinline__ void fold_antisym(T *acc)
{
  acc[11] = -(acc[3] + acc[7]);
  acc[4] += acc[14];
  acc[5] -= acc[13];
  acc[6] -= acc[14];
  acc[8] += acc[12];
  acc[9] += acc[13];
  acc[10] -= acc[12];
}

// TSIG: the core size comes from the TARGET body instead of the source.  That is the
// transposed near-field kernel used by the adjoint (a particle's own sigma, with the
// particle now on the target side).
//
// One workgroup per unit (near_units.hpp): the list entries [q0, q1) of target leaf w.  A leaf whose
// list is one unit is stored directly; a leaf cut into several units leaves each unit's sums
// (12 rows of nt doubles) at part + 12 * row, and k_p2p_reduce adds them in unit order, so the
// result does not depend on which unit runs when.
//
// Chunks: 64 lanes stage 128 sources at a time (two per lane, both searches and all loads in
// flight together) and 256 lanes 256.
//
// Bound by VALU issue: 47 lane-instructions a pair in FP32, 82 in FP64 while x < X64 (62 of them
// multiply-adds).  Units and chunks against one workgroup per leaf, and in FP64 the polynomial pair
// factors against erf, exp, sqrt and divisions: 1M two rings FP64 10.2 -> 4.4 ms (1.54e9 pairs), 8k
// ring FP64 1.34 -> 0.075 ms, 60k cube mixed 2.65 -> 1.18 ms; 4M two rings
// mixed 10.0 -> 9.6 ms.
template <bool MIXED, bool WITH_J, bool TSIG, int BLK>
__global__ __launch_bounds__(BLK) __attribute__((amdgpu_waves_per_eu(MIXED ? 5 : 3))) void k_p2p(
    const int4 *__restrict__ units, const int32_t *__restrict__ leaves, const int32_t *__restrict__ tbody,
    const int32_t *__restrict__ tnbody, const double *__restrict__ tcx, const double *__restrict__ tcy,
    const double *__restrict__ tcz, const int32_t *__restrict__ src, const int32_t *__restrict__ sbody,
    const int32_t *__restrict__ snbody, const double *__restrict__ tst, int64_t tcap, const double *__restrict__ sst,
    int64_t scap, double *__restrict__ out, int64_t ocap, double *__restrict__ part)
{
  // One LDS buffer holds the staged sources during the pair loops (two float4 or two double4 an
  // entry) and the partial sums of the splits after them (12 doubles per lane).  CH entries are
  // staged; up to ENT are read, those past the chunk are padding (2 S <= CH, see near_splits: at
  // most 2 S ceil(CH / 2 S) <= 3/2 CH entries).
  constexpr int CH = BLK == 64 ? 128 : 256, ENT = CH + CH / 2, PER = CH / BLK, ESZ = MIXED ? 32 : 64;
  constexpr int SMEM = ENT * ESZ > 96 * BLK ? ENT * ESZ : 96 * BLK;
  __shared__ __align__(16) unsigned char smem[SMEM];
  __shared__ int pref[SEG + 1], lb[SEG];
  using T  = typename std::conditional<MIXED, float, double>::type;
  using T4 = typename std::conditional<MIXED, float4, double4>::type;
  T4     *sv  = reinterpret_cast<T4 *>(smem);
  double *red = reinterpret_cast<double *>(smem);
  const int4 un = units[blockIdx.x];
  const int  t = leaves[un.x], tb = tbody[t], nt = tnbody[t], q0 = un.y, q1 = un.z, prow = un.w;
  const int  lane = threadIdx.x;
  // lanes = (target ti) x (source split si): ntp targets per pass (near_targets_per_pass); the
  // BLK - ntp * S lanes left over take the first split's sources and are dropped
  const int    ntp = near_targets_per_pass<BLK>(nt), S = near_splits<BLK>(ntp), ti = lane % ntp, si = lane / ntp;
  const bool   lane_on = si < S;
  // offsets from the target leaf's centre (mixed: formed in FP64, then rounded to FP32); FP64 keeps
  // the absolute coordinates
  const double cxt = MIXED ? tcx[t] : 0.0, cyt = MIXED ? tcy[t] : 0.0, czt = MIXED ? tcz[t] : 0.0;
  for (int c0 = 0; c0 < nt; c0 += ntp) {
    const int     i     = c0 + ti;
    const bool    valid = lane_on && i < nt;
    const int64_t bi = tb + (valid ? i : 0);
    const T rxi = (T)(tst[(F_X + 0) * tcap + bi] - cxt), ryi = (T)(tst[(F_X + 1) * tcap + bi] - cyt),
            rzi = (T)(tst[(F_X + 2) * tcap + bi] - czt);
    // target-sigma constants (TSIG only)
    const double tsg = TSIG ? tst[F_SIG * tcap + bi] : 1.0;
    const double tqq = MIXED ? 0.5 / (tsg * tsg) : core_q64(tsg), tc1 = pow32(tqq) * INV_4PI;
    const T      t_q = (T)tqq, t_c1 = (T)tc1, t_c2 = (T)(2.0 * tqq * tc1);
    double       acc[MIXED ? 12 : 15];
    for (int k = 0; k < (MIXED ? 12 : 15); k++) acc[k] = 0.0;
    for (int g0 = q0; g0 < q1; g0 += SEG) {
      const int nseg = min(SEG, q1 - g0);
      __syncthreads();
      for (int k = lane; k < nseg; k += BLK) {
        const int sl = src[g0 + k];
        lb[k]        = sbody[sl];
        pref[k]      = snbody[sl];
      }
      __syncthreads();
      if (lane < 64) lds_prefix(pref, pref, nseg);
      __syncthreads();
      const int total = pref[nseg];
      for (int j0 = 0; j0 < total; j0 += CH) {
        const int cnt = min(CH, total - j0);
        const int T2  = 2 * ((cnt + 2 * S - 1) / (2 * S));  // entries per lane: si, si + S, ...
        double    x[PER], y[PER], z[PER], sg[PER], ax[PER], ay[PER], az[PER];
#pragma unroll
        for (int p = 0; p < PER; p++) {
          // entries past the chunk load its last one again and are stored as padding
          const int64_t bj = list_body(pref, lb, nseg, j0 + min(lane + p * BLK, cnt - 1));
          x[p] = sst[(F_X + 0) * scap + bj], y[p] = sst[(F_X + 1) * scap + bj], z[p] = sst[(F_X + 2) * scap + bj];
          sg[p] = sst[F_SIG * scap + bj];
          ax[p] = sst[(F_A + 0) * scap + bj], ay[p] = sst[(F_A + 1) * scap + bj], az[p] = sst[(F_A + 2) * scap + bj];
        }
        // Entries of no strength past the chunk: every lane runs the same trip count.  Their offset
        // and q put x = |r - (1024, 0, 0)|^2 / 2^20 near 1 for any target within a few hundred units
        // of the leaf centre, so they stay on the pair loop's common path (a pad at x = 0 would take
        // its coincident-pair test); TSIG takes q from the target, where a pad at the centre gives
        // x = |r|^2 q of the same order as the real pairs.
        T4 padA, padB;
        padA.x = (T)(TSIG ? 0.0 : 1024.0) + (T)(MIXED ? 0.0 : tcx[t]), padA.y = (T)(MIXED ? 0.0 : tcy[t]);
        padA.z = (T)(MIXED ? 0.0 : tcz[t]), padA.w = (T)0x1p-20;
        padB.x = padB.y = padB.z = padB.w = (T)0.0;
#pragma unroll
        for (int p = 0; p < PER; p++) {
          const int e = lane + p * BLK;
          if (e < cnt) {
            // (offset, q) and (alpha c1, 2 q) with q = 1 / (2 sigma^2), c1 = q^{3/2} / (4 pi): then
            // f1 = G(x) and f2 = 2 q G'(x) for the scaled strength.  TSIG keeps alpha as is.
            const double qq = MIXED ? 0.5 / (sg[p] * sg[p]) : core_q64(sg[p]), c1 = TSIG ? 1.0 : pow32(qq) * INV_4PI;
            T4           A, B;
            A.x = (T)(x[p] - cxt), A.y = (T)(y[p] - cyt), A.z = (T)(z[p] - czt), A.w = (T)qq;
            B.x = (T)(ax[p] * c1), B.y = (T)(ay[p] * c1), B.z = (T)(az[p] * c1), B.w = (T)(2.0 * qq);
            sv[2 * e] = A, sv[2 * e + 1] = B;
          }
        }
        for (int e = cnt + lane; e < T2 * S; e += BLK) sv[2 * e] = padA, sv[2 * e + 1] = padB;
        __syncthreads();
        const T4 *ps = sv + 2 * (lane_on ? si : 0);
        if constexpr (MIXED) {
          // lane (ti, si) takes entries si, si + S, ... two per step.
          float fa[15];
          // FP32 partial sums cover at most FLUSH entries per lane before they go into the FP64 sums
          constexpr int FLUSH = 64;
          for (int k0 = 0; k0 < T2; k0 += FLUSH) {
            for (int k = 0; k < 15; k++) fa[k] = 0.f;
            for (int k = k0; k < min(T2, k0 + FLUSH); k += 2, ps += 4 * S) {
              const float4 A0 = ps[0], B0 = ps[1], A1 = ps[2 * S], B1 = ps[2 * S + 1];
              const float  dx0 = rxi - A0.x, dy0 = ryi - A0.y, dz0 = rzi - A0.z;
              const float  dx1 = rxi - A1.x, dy1 = ryi - A1.y, dz1 = rzi - A1.z;
              const float  r20 = dx0 * dx0 + dy0 * dy0 + dz0 * dz0, r21 = dx1 * dx1 + dy1 * dy1 + dz1 * dz1;
              const float  q0 = TSIG ? t_q : A0.w, q1 = TSIG ? t_q : A1.w;
              const float  tq0 = fmaf(r20, q0, -1.0f), tq1 = fmaf(r21, q1, -1.0f);  // x - 1
              float        G0, Gp0, G1, Gp1;  // G(x) and G'(x) of both pairs
              g_near(tq0, tq1, G0, Gp0, G1, Gp1);
              // x >= 2 (t >= 1) takes the far form, and a coincident pair (R^2 = 0, so t = -1
              // exactly) is skipped (multipoleKernels.hpp:242).  t >= -1 always, so one test
              // |t| >= 1 over both pairs sends the rare steps that need either fix-up off the
              // common path.
              if (fmaxf(fabsf(tq0), fabsf(tq1)) >= XPOLY - 1.0f) {
                if (fmaxf(tq0, tq1) >= XPOLY - 1.0f) {  // lanes with a far pair take both far forms
                  float Gf0, Gpf0, Gf1, Gpf1;
                  g_far(r20 * q0, Gf0, Gpf0);
                  g_far(r21 * q1, Gf1, Gpf1);
                  if (tq0 >= XPOLY - 1.0f) G0 = Gf0, Gp0 = Gpf0;
                  if (tq1 >= XPOLY - 1.0f) G1 = Gf1, Gp1 = Gpf1;
                }
                // only the f1 alpha terms of J survive a zero dX, so zeroing f1 is enough
                if (r20 == 0.0f) G0 = 0.0f;
                if (r21 == 0.0f) G1 = 0.0f;
              }
              const float f10 = TSIG ? G0 * t_c1 : G0;
              const float f11 = TSIG ? G1 * t_c1 : G1;
              accumulate_pair(fa, dx0, dy0, dz0, B0.x, B0.y, B0.z, f10, Gp0 * (TSIG ? t_c2 : B0.w), WITH_J);
              accumulate_pair(fa, dx1, dy1, dz1, B1.x, B1.y, B1.z, f11, Gp1 * (TSIG ? t_c2 : B1.w), WITH_J);
            }
            if (WITH_J) fold_antisym(fa);
            for (int k = 0; k < (WITH_J ? 12 : 3); k++) acc[k] += (double)fa[k];
          }
        } else {
          for (int k = 0; k < T2; k += 2, ps += 4 * S) {
            const double4 A0 = ps[0], B0 = ps[1], A1 = ps[2 * S], B1 = ps[2 * S + 1];
            const double  dx0 = rxi - A0.x, dy0 = ryi - A0.y, dz0 = rzi - A0.z;
            const double  dx1 = rxi - A1.x, dy1 = ryi - A1.y, dz1 = rzi - A1.z;
            const double  r20 = dx0 * dx0 + dy0 * dy0 + dz0 * dz0, r21 = dx1 * dx1 + dy1 * dy1 + dz1 * dz1;
            double        G0, Gp0, G1, Gp1;
            g64_pair2(r20, r21, TSIG ? t_q : A0.w, TSIG ? t_q : A1.w, G0, Gp0, G1, Gp1);
            const double f10 = TSIG ? G0 * t_c1 : G0;
            const double f11 = TSIG ? G1 * t_c1 : G1;
            accumulate_pair(acc, dx0, dy0, dz0, B0.x, B0.y, B0.z, f10, Gp0 * (TSIG ? t_c2 : B0.w), WITH_J);
            accumulate_pair(acc, dx1, dy1, dz1, B1.x, B1.y, B1.z, f11, Gp1 * (TSIG ? t_c2 : B1.w), WITH_J);
          }
        }
        __syncthreads();
      }
    }
    if constexpr (!MIXED && WITH_J) fold_antisym(acc);
    // Sum of the S splits (lanes t + q * ntp) in split order, through LDS: the lanes then take
    // (field, target) pairs, consecutive targets in consecutive lanes.
    constexpr int NK = WITH_J ? 12 : 3;
    const int     np = min(ntp, nt - c0);
    __syncthreads();
    for (int k = 0; k < NK; k++) red[k * BLK + lane] = acc[k];
    __syncthreads();
    for (int o = lane; o < NK * np; o += BLK) {
      const int k = o / np, tt = o - k * np;
      double    v = red[k * BLK + tt];
      for (int q = 1; q < S; q++) v += red[k * BLK + tt + q * ntp];
      if (prow >= 0) part[((int64_t)prow * 12 + (int64_t)k * nt) + c0 + tt] = v;
      else out[(k < 3 ? F_U + k : F_J + k - 3) * ocap + tb + c0 + tt] = -v;
    }
  }
}

// O(m n) direct sum, FP64.  Output: u (m,3), J (m,9) and, when target strengths are given, the
// classic stretching J.alpha_t (the quantity exafmm::direct produces, traverse.hpp:88-98).
//
// A workgroup of 1024 lanes takes NT targets against all sources: lanes = (target) x (1024 / NT
// source splits), sources staged 1024 at a time, the next chunk's loads in flight during the pair
// loop, the splits added in order through LDS.  NT is the largest power of two that still gives
// DIRECT_BLOCKS workgroups: a target per lane and no splits left 4096 targets on 16 of 256 CUs
// (109.7 ms against 200k sources).  Fewer targets per workgroup stage each source more often: at
// NT = 16 the staging is 1 of 17 lane-steps.  No workspace: uvlm_direct_noalloc runs it too.
constexpr int DIRECT_LANES = 1024, DIRECT_BLOCKS = 256;
template <bool WITH_J>
__global__ __launch_bounds__(DIRECT_LANES) void k_direct(int NT, int64_t m, const double *__restrict__ xt,
                                                         const double *__restrict__ at,
                                                         const double *__restrict__ sst, int64_t scap, int64_t n,
                                                         double *__restrict__ u, double *__restrict__ J,
                                                         double *__restrict__ dadt)
{
  __shared__ __align__(32) unsigned char smem[64 * DIRECT_LANES];
  // (x, q), (alpha, c1), q and c1 as in k_p2p; alpha unscaled, so a separation along it still gives 0
  double4      *sv  = reinterpret_cast<double4 *>(smem);
  double       *red = reinterpret_cast<double *>(smem);   // half of the 12 sums at a time
  const int     tid = threadIdx.x, ti = tid & (NT - 1), si = tid / NT, S = DIRECT_LANES / NT;
  const int64_t i0 = blockIdx.x * (int64_t)NT, i = min(i0 + ti, m - 1);
  const double  xi = xt[3 * i], yi = xt[3 * i + 1], zi = xt[3 * i + 2];
  double        acc[15];
  for (int k = 0; k < 15; k++) acc[k] = 0.0;
  double v[7];
  auto   load = [&](int64_t j) {
    j = min(j, n - 1);
    for (int d = 0; d < 3; d++) v[d] = sst[(F_X + d) * scap + j], v[3 + d] = sst[(F_A + d) * scap + j];
    v[6] = sst[F_SIG * scap + j];
  };
  load(tid);
  for (int64_t j0 = 0; j0 < n; j0 += DIRECT_LANES) {
    const int cnt = (int)min<int64_t>(DIRECT_LANES, n - j0);
    const int T2  = 2 * ((cnt + 2 * S - 1) / (2 * S));  // entries per lane; T2 * S <= DIRECT_LANES as NT is even
    double4   A, B;
    if (tid < cnt) {
      const double qq = core_q64(v[6]);
      A.x = v[0], A.y = v[1], A.z = v[2], A.w = qq;
      B.x = v[3], B.y = v[4], B.z = v[5], B.w = pow32(qq) * INV_4PI;
    } else {  // no strength, x near 1 for targets within some hundred units (see k_p2p)
      A.x = v[0] + 1024.0, A.y = v[1], A.z = v[2], A.w = 0x1p-20;
      B.x = B.y = B.z = B.w = 0.0;
    }
    sv[2 * tid] = A, sv[2 * tid + 1] = B;
    __syncthreads();
    if (j0 + DIRECT_LANES < n) load(j0 + DIRECT_LANES + tid);
    const double4 *ps = sv + 2 * si;
    for (int k = 0; k < T2; k += 2, ps += 4 * S) {
      const double4 A0 = ps[0], B0 = ps[1], A1 = ps[2 * S], B1 = ps[2 * S + 1];
      const double  dx0 = xi - A0.x, dy0 = yi - A0.y, dz0 = zi - A0.z;
      const double  dx1 = xi - A1.x, dy1 = yi - A1.y, dz1 = zi - A1.z;
      const double  r20 = dx0 * dx0 + dy0 * dy0 + dz0 * dz0, r21 = dx1 * dx1 + dy1 * dy1 + dz1 * dz1;
      double        G0, Gp0, G1, Gp1;
      g64_pair2(r20, r21, A0.w, A1.w, G0, Gp0, G1, Gp1);
      accumulate_pair(acc, dx0, dy0, dz0, B0.x, B0.y, B0.z, G0 * B0.w, 2.0 * Gp0 * (A0.w * B0.w), WITH_J);
      accumulate_pair(acc, dx1, dy1, dz1, B1.x, B1.y, B1.z, G1 * B1.w, 2.0 * Gp1 * (A1.w * B1.w), WITH_J);
    }
    __syncthreads();
  }
  if (WITH_J) fold_antisym(acc);
  // the splits of each (field, target), six fields at a time; lanes (field, target)
  for (int h = 0; h < (WITH_J ? 2 : 1); h++) {
    for (int k = 0; k < 6; k++) red[k * DIRECT_LANES + tid] = acc[h ? 6 + k : k];
    __syncthreads();
    for (int o = tid; o < (WITH_J ? 6 : 3) * NT; o += DIRECT_LANES) {
      const int k = o / NT, t = o & (NT - 1);
      double    w = 0.0;
      for (int q = 0; q < S; q++) w += red[k * DIRECT_LANES + q * NT + t];
      const int f = 6 * h + k;
      if (i0 + t < m) {
        if (f < 3) u[3 * (i0 + t) + f] = -w;
        else if (J) J[9 * (i0 + t) + f - 3] = -w;
      }
      // kept for the stretching: this lane's sum goes back where it came from, split 0
      red[k * DIRECT_LANES + t] = w;
    }
    __syncthreads();
    if (WITH_J && dadt && at && tid < NT && i0 + tid < m) {
      const double *a = at + 3 * (i0 + tid);
      if (h == 0) acc[0] = red[3 * DIRECT_LANES + tid] * a[0] + red[4 * DIRECT_LANES + tid] * a[1] + red[5 * DIRECT_LANES + tid] * a[2];
      else {
        double *o = dadt + 3 * (i0 + tid);
        o[0] = -acc[0];
        for (int r = 0; r < 2; r++)
          o[1 + r] = -(red[3 * r * DIRECT_LANES + tid] * a[0] + red[(3 * r + 1) * DIRECT_LANES + tid] * a[1] +
                       red[(3 * r + 2) * DIRECT_LANES + tid] * a[2]);
      }
    }
    __syncthreads();
  }
}

}  // namespace

void direct(hipStream_t s, int64_t m, const double *xt, const double *at, const double *sst, int64_t scap, int64_t n,
            double *u, double *J, double *dadt)
{
  if (m <= 0) return;
  int NT = 64;
  while (NT > 2 && (m + NT - 1) / NT < DIRECT_BLOCKS) NT /= 2;
  const int nb = (int)((m + NT - 1) / NT);
  if (J || dadt) k_direct<true><<<nb, DIRECT_LANES, 0, s>>>(NT, m, xt, at, sst, scap, n, u, J, dadt);
  else k_direct<false><<<nb, DIRECT_LANES, 0, s>>>(NT, m, xt, at, sst, scap, n, u, J, dadt);
  UVLM_LAUNCH_CHECK();
}

// Totals of the near-field units (near_units.hpp).
enum { NU_INTER = 0, NU_WORK, NU_ROWWORK, NU_UNITS, NU_ROWS, NU_MULTI, NU_WIDE, NU_COUNT };
static_assert(UNIT_COUNTERS + NU_COUNT <= N_COUNTERS, "near-field unit totals");

__global__ void k_units_clear(unsigned long long *__restrict__ cnt)
{
  if (threadIdx.x < NU_COUNT) cnt[threadIdx.x] = 0;
}

// work[w] (lane steps) of each target leaf and the sums over all: interactions, work, targets times
// work.  One wavefront per leaf at a time, lanes over its list; at most UNITS_WORK_BLOCKS blocks keep
// the same-address atomics few.
constexpr int UNITS_WORK_BLOCKS = 512;
__global__ __launch_bounds__(256) void k_units_work(const int32_t *__restrict__ leaves, int64_t nleaf,
                                                    int64_t max_leaf, int64_t nsleaf, double narrow, int lanes,
                                                    const unsigned long long *__restrict__ np2p,
                                                    const int32_t *__restrict__ tnbody,
                                                    const int32_t *__restrict__ off, const int32_t *__restrict__ src,
                                                    const int32_t *__restrict__ snbody, uint32_t *__restrict__ work,
                                                    unsigned long long *__restrict__ cnt)
{
  __shared__ unsigned long long sum[3][4];
  // mean pairs a leaf (cell 0 is the root: all bodies)
  const double pairs = (double)*np2p / nleaf * ((double)tnbody[0] / nleaf) * ((double)snbody[0] / nsleaf);
  const bool   wide  = units_wide(nleaf, max_leaf, pairs, narrow, lanes);
  if (blockIdx.x == 0 && threadIdx.x == 0) cnt[NU_WIDE] = wide;
  const int          lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  unsigned long long inter = 0, all = 0, rows = 0;
  for (int64_t w = blockIdx.x * 4ll + wv; w < nleaf; w += gridDim.x * 4ll) {
    const int t = leaves[w], nt = tnbody[t], q1 = off[t + 1];
    unsigned  ns = 0;
#pragma unroll 4  // four gathers in flight: 29 -> 13 us for lists of thousands (4096 probes of 200003 bodies)
    for (int q = off[t] + lane; q < q1; q += 64) ns += (unsigned)snbody[src[q]];
    for (int o = 32; o > 0; o >>= 1) ns += __shfl_xor(ns, o, 64);
    const int ntp = wide ? near_targets_per_pass<256>(nt) : near_targets_per_pass<64>(nt);
    const int S   = wide ? near_splits<256>(ntp) : near_splits<64>(ntp);
    const unsigned long long steps = ((unsigned long long)ns * ((nt + ntp - 1) / ntp) + S - 1) / S;
    const uint32_t           wk    = (uint32_t)min(steps, 0xffffffffull);
    if (lane == 0) work[w] = wk;
    inter += (unsigned long long)nt * ns;
    all += wk;
    rows += (unsigned long long)nt * wk;
  }
  if (lane == 0) sum[0][wv] = inter, sum[1][wv] = all, sum[2][wv] = rows;
  __syncthreads();
  if (threadIdx.x < 3) {
    unsigned long long v = 0;
    for (int k = 0; k < 4; k++) v += sum[threadIdx.x][k];
    if (v) atomicAdd(&cnt[threadIdx.x], v);
  }
}

// Units (w, first entry, end, row of the partial sums or -1) and the leaves cut into several
// (w, first row, units).  Ranges are reserved once per block.
__global__ __launch_bounds__(256) void k_units_fill(const int32_t *__restrict__ leaves, int64_t nleaf,
                                                    const int32_t *__restrict__ tnbody,
                                                    const int32_t *__restrict__ off,
                                                    const uint32_t *__restrict__ work, uint64_t rows,
                                                    unsigned long long *__restrict__ cnt, int4 *__restrict__ units,
                                                    int4 *__restrict__ multi)
{
  __shared__ unsigned long long tot[4][3], base[3];
  const int64_t            w    = blockIdx.x * 256ll + threadIdx.x;
  const int                lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint64_t           lim = units_limit(cnt[NU_WORK], cnt[NU_ROWWORK], rows);
  int                      nu = 0, q0 = 0, len = 0, nt = 0;  // no units past the last leaf
  if (w < nleaf) {
    const int t = leaves[w];
    nt = tnbody[t], q0 = off[t], len = off[t + 1] - q0;
    nu = units_of_leaf(work[w], len, lim);
  }
  // exclusive prefix sums over the block of units, rows and cut leaves
  unsigned long long v[3] = {(unsigned long long)nu, nu > 1 ? (unsigned long long)nu * nt : 0, nu > 1 ? 1ull : 0}, ex[3];
  for (int c = 0; c < 3; c++) {
    unsigned long long x = v[c];
    for (int o = 1; o < 64; o <<= 1) {
      const unsigned long long u = __shfl_up(x, o, 64);
      if (lane >= o) x += u;
    }
    if (lane == 63) tot[wv][c] = x;
    ex[c] = x - v[c];
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    unsigned long long sum = 0;
    for (int k = 0; k < 4; k++) sum += tot[k][threadIdx.x];
    base[threadIdx.x] = sum ? atomicAdd(&cnt[NU_UNITS + threadIdx.x], sum) : 0;
  }
  __syncthreads();
  for (int c = 0; c < 3; c++) {
    ex[c] += base[c];
    for (int k = 0; k < wv; k++) ex[c] += tot[k][c];
  }
  if (nu > 1 && w < nleaf) multi[ex[2]] = make_int4((int)w, (int)ex[1], nu, 0);
  // the block's units, written by all its lanes (a probe tree's few leaves have hundreds each)
  __shared__ int first[257], row[256], q0s[256], lens[256], nts[256];
  first[threadIdx.x] = (int)(ex[0] - base[0]);
  row[threadIdx.x] = (int)ex[1], q0s[threadIdx.x] = q0, lens[threadIdx.x] = len, nts[threadIdx.x] = nt;
  if (threadIdx.x == 255) first[256] = first[255] + nu;
  __syncthreads();
  for (int u = threadIdx.x; u < first[256]; u += 256) {
    int lo = 0, hi = 255;  // the last leaf with first <= u (leaves past the end have no units)
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (first[mid] <= u) lo = mid;
      else hi = mid - 1;
    }
    const int n = first[lo + 1] - first[lo], j = u - first[lo], ln = lens[lo];
    units[base[0] + u] = make_int4((int)(blockIdx.x * 256 + lo), q0s[lo] + units_first(ln, j, n),
                                   q0s[lo] + units_first(ln, j + 1, n), n > 1 ? row[lo] + j * nts[lo] : -1);
  }
}

// Sums of the leaves cut into several units, units in order, stored as k_p2p stores a single one.
template <bool WITH_J>
__global__ __launch_bounds__(256) void k_p2p_reduce(const int4 *__restrict__ multi, const int32_t *__restrict__ leaves,
                                                    const int32_t *__restrict__ tbody,
                                                    const int32_t *__restrict__ tnbody,
                                                    const double *__restrict__ part, double *__restrict__ out,
                                                    int64_t ocap)
{
  const int4    m = multi[blockIdx.x];
  const int     t = leaves[m.x], tb = tbody[t], nt = tnbody[t];
  const double *p = part + (int64_t)m.y * 12;
  for (int o = threadIdx.x; o < (WITH_J ? 12 : 3) * nt; o += 256) {
    const int k = o / nt;
    double    v = 0.0;
#pragma unroll 16  // 16 rows in flight (4: 22 us for the same probes, 16: 13)
    for (int u = 0; u < m.z; u++) v += p[(int64_t)u * 12 * nt + o];
    out[(k < 3 ? F_U + k : F_J + k - 3) * ocap + tb + (o - k * nt)] = -v;
  }
}

// Gaussian near-field sums over the P2P lists, FP64 (the viscous and vorticity kernels of
// multipoleKernels.hpp:343-450).
//  GAUSS_PSE : dadt_i += prefix * sum_j (vol_i a_j - vol_j a_i) e^{-R^2 / (2 s_ij^2)} / s_ij^5,
//              s_ij^2 = sigma_i^2 + sigma_j^2, vol = 4/3 pi sigma^3, pairs with R^2 = 0 skipped
//  GAUSS_VORT: out[field + d]_i -= sum_j a_j,d e^{-R^2 / (2 sigma_j^2)} / ((2 pi)^{3/2} sigma_j^3)
// Units, chunks, lanes and the sum of the splits are k_p2p's; sums in a fixed order.  Bound by VALU
// issue: about 55 lane-instructions a pair (PSE: the exponential 18, the reciprocal root of s_ij^2
// 7).  One lane per target with library exp, sqrt and two divisions took 2.6 ms for the 100k two
// rings (136e6 pairs, up to 100 bodies a leaf).
enum { GAUSS_PSE = 0, GAUSS_VORT = 1 };
template <int MODE, int BLK>
__global__ __launch_bounds__(BLK) void k_gauss(const int4 *__restrict__ units, const int32_t *__restrict__ leaves,
                                               const int32_t *__restrict__ tbody, const int32_t *__restrict__ tnbody,
                                               const int32_t *__restrict__ src, const int32_t *__restrict__ sbody,
                                               const int32_t *__restrict__ snbody, const double *__restrict__ tst,
                                               int64_t tcap, const double *__restrict__ sst, int64_t scap,
                                               double *__restrict__ out, int64_t ocap, int field, double prefix,
                                               double *__restrict__ part)
{
  constexpr int CH = BLK == 64 ? 128 : 256, ENT = CH + CH / 2, PER = CH / BLK;
  __shared__ __align__(32) unsigned char smem[ENT * 64];
  __shared__ int pref[SEG + 1], lb[SEG];
  double4 *sv  = reinterpret_cast<double4 *>(smem);  // (x, sigma^2 or q), (alpha, vol) or (alpha c, 0)
  double  *red = reinterpret_cast<double *>(smem);
  const int4 un = units[blockIdx.x];
  const int  t = leaves[un.x], tb = tbody[t], nt = tnbody[t], q0 = un.y, q1 = un.z, prow = un.w;
  const int  lane = threadIdx.x;
  const int  ntp = near_targets_per_pass<BLK>(nt), S = near_splits<BLK>(ntp), ti = lane % ntp, si = lane / ntp;
  const bool lane_on = si < S;
  for (int c0 = 0; c0 < nt; c0 += ntp) {
    const int     i  = c0 + ti;
    const int64_t bi = tb + (lane_on && i < nt ? i : 0);
    const double  xi = tst[(F_X + 0) * tcap + bi], yi = tst[(F_X + 1) * tcap + bi], zi = tst[(F_X + 2) * tcap + bi];
    double        s2i = 0.0, voli = 0.0, ai[3] = {0.0, 0.0, 0.0};
    if (MODE == GAUSS_PSE) {
      const double sg = tst[F_SIG * tcap + bi];
      s2i  = sg * sg;
      voli = 4. / 3. * M_PI * sg * sg * sg;
      for (int d = 0; d < 3; d++) ai[d] = tst[(F_A + d) * tcap + bi];
    }
    double acc[3] = {0.0, 0.0, 0.0};
    auto   sep  = [&](const double4 &A) {
      const double dx = xi - A.x, dy = yi - A.y, dz = zi - A.z;
      return dx * dx + dy * dy + dz * dz;
    };
    auto add = [&](const double4 &A, const double4 &B, double R2, double r, double x) {
      if (MODE == GAUSS_PSE) {
        const double o2 = r * r, e = R2 == 0.0 ? 0.0 : exp64_neg(x, c_exp64) * (o2 * o2 * r);
        acc[0] = fma(voli * B.x - B.w * ai[0], e, acc[0]);
        acc[1] = fma(voli * B.y - B.w * ai[1], e, acc[1]);
        acc[2] = fma(voli * B.z - B.w * ai[2], e, acc[2]);
      } else {
        const double e = exp64_neg(x, c_exp64);
        acc[0] = fma(B.x, e, acc[0]);
        acc[1] = fma(B.y, e, acc[1]);
        acc[2] = fma(B.z, e, acc[2]);
      }
    };
    auto pairs = [&](const double4 &A0, const double4 &B0, const double4 &A1, const double4 &B1) {
      const double R0 = sep(A0), R1 = sep(A1);
      double       r0 = 0.0, r1 = 0.0, x0, x1;  // PSE: 1 / s_ij
      if (MODE == GAUSS_PSE) {
        r0 = rsqrt64(s2i + A0.w), r1 = rsqrt64(s2i + A1.w);
        x0 = 0.5 * R0 * (r0 * r0), x1 = 0.5 * R1 * (r1 * r1);
      } else x0 = R0 * A0.w, x1 = R1 * A1.w;
      x0 = exp64_arg(x0), x1 = exp64_arg(x1);
      add(A0, B0, R0, r0, x0);
      add(A1, B1, R1, r1, x1);
    };
    for (int g0 = q0; g0 < q1; g0 += SEG) {
      const int nseg = min(SEG, q1 - g0);
      __syncthreads();
      for (int k = lane; k < nseg; k += BLK) {
        const int sl = src[g0 + k];
        lb[k]        = sbody[sl];
        pref[k]      = snbody[sl];
      }
      __syncthreads();
      if (lane < 64) lds_prefix(pref, pref, nseg);
      __syncthreads();
      const int total = pref[nseg];
      for (int j0 = 0; j0 < total; j0 += CH) {
        const int cnt = min(CH, total - j0);
        const int T2  = 2 * ((cnt + 2 * S - 1) / (2 * S));
        double    v[PER][7];
#pragma unroll
        for (int p = 0; p < PER; p++) {
          const int64_t bj = list_body(pref, lb, nseg, j0 + min(lane + p * BLK, cnt - 1));
          for (int d = 0; d < 3; d++) v[p][d] = sst[(F_X + d) * scap + bj], v[p][3 + d] = sst[(F_A + d) * scap + bj];
          v[p][6] = sst[F_SIG * scap + bj];
        }
#pragma unroll
        for (int p = 0; p < PER; p++) {
          const int e = lane + p * BLK;
          if (e < cnt) {
            const double sg = v[p][6], S2 = 2.0 * sg * sg;
            double       c  = MODE == GAUSS_PSE ? 1.0 : (INV_PI * INV_SQRTPI * 0.70710678118654752440) / S2 / sg;
            if (MODE == GAUSS_VORT && S2 > 0.0) c = fmax(fmin(c, 1e290), -1e290);  // no infinity times e = 0
            double4      A, B;
            A.x = v[p][0], A.y = v[p][1], A.z = v[p][2], A.w = MODE == GAUSS_PSE ? sg * sg : 1.0 / S2;
            B.x = v[p][3] * c, B.y = v[p][4] * c, B.z = v[p][5] * c;
            B.w = MODE == GAUSS_PSE ? 4. / 3. * M_PI * sg * sg * sg : 0.0;
            sv[2 * e] = A, sv[2 * e + 1] = B;
          }
        }
        // entries of no strength and no volume past the chunk
        double4 pad;
        pad.x = pad.y = pad.z = pad.w = 1.0;
        double4 none;
        none.x = none.y = none.z = none.w = 0.0;
        for (int e = cnt + lane; e < T2 * S; e += BLK) sv[2 * e] = pad, sv[2 * e + 1] = none;
        __syncthreads();
        const double4 *ps = sv + 2 * (lane_on ? si : 0);
        for (int k = 0; k < T2; k += 2, ps += 4 * S) pairs(ps[0], ps[1], ps[2 * S], ps[2 * S + 1]);
        __syncthreads();
      }
    }
    const int np = min(ntp, nt - c0);
    __syncthreads();
    for (int d = 0; d < 3; d++) red[d * BLK + lane] = acc[d];
    __syncthreads();
    for (int o = lane; o < 3 * np; o += BLK) {
      const int d = o / np, tt = o - d * np;
      double    v = red[d * BLK + tt];
      for (int q = 1; q < S; q++) v += red[d * BLK + tt + q * ntp];
      if (prow >= 0) part[(int64_t)prow * 12 + (int64_t)d * nt + c0 + tt] = v;
      else if (MODE == GAUSS_PSE) out[(F_DADT + d) * ocap + tb + c0 + tt] += v * prefix;
      else out[(field + d) * ocap + tb + c0 + tt] -= v;
    }
  }
}

template <int MODE>
__global__ __launch_bounds__(256) void k_gauss_reduce(const int4 *__restrict__ multi,
                                                      const int32_t *__restrict__ leaves,
                                                      const int32_t *__restrict__ tbody,
                                                      const int32_t *__restrict__ tnbody,
                                                      const double *__restrict__ part, double *__restrict__ out,
                                                      int64_t ocap, int field, double prefix)
{
  const int4    m = multi[blockIdx.x];
  const int     t = leaves[m.x], tb = tbody[t], nt = tnbody[t];
  const double *p = part + (int64_t)m.y * 12;
  for (int o = threadIdx.x; o < 3 * nt; o += 256) {
    const int d = o / nt;
    double    v = 0.0;
#pragma unroll 4
    for (int u = 0; u < m.z; u++) v += p[(int64_t)u * 12 * nt + o];
    if (MODE == GAUSS_PSE) out[(F_DADT + d) * ocap + tb + (o - d * nt)] += v * prefix;
    else out[(field + d) * ocap + tb + (o - d * nt)] -= v;
  }
}

// Units of the P2P list `l` (np2p entries, on the device) of target tree tt against source tree st
// (see k_units_work), and the number of near-field interactions.  cleared: the units' counters are
// zero.  rows: the rows of partial sums they may have.
void near_units_enqueue(hipStream_t s, Scratch &sc, const Tree &tt, const Tree &st, int64_t max_leaf,
                        const unsigned long long *np2p, bool cleared, Lists &l, uint64_t rows)
{
  if (tt.nleaf == 0) return;
  sc.unit_work.reserve(4 * tt.nleaf);
  unsigned long long *cnt = sc.counters.as<unsigned long long>() + UNIT_COUNTERS;
  l.units.reserve(sizeof(int4) * units_bound(tt.nleaf));
  l.multi.reserve(sizeof(int4) * units_multi_bound(tt.nleaf));
  const int32_t *lv = tt.leaves.as<int32_t>(), *tn = tt.nbody.as<int32_t>();
  const int32_t *off = l.p2p_off.as<int32_t>();
  if (!cleared) k_units_clear<<<1, 64, 0, s>>>(cnt);
  k_units_work<<<(int)std::min<int64_t>(UNITS_WORK_BLOCKS, (tt.nleaf + 3) / 4), 256, 0, s>>>(
      lv, tt.nleaf, max_leaf, st.nleaf, sc.near_narrow, sc.near_lanes, np2p, tn, off, l.p2p_src.as<int32_t>(), st.nbody.as<int32_t>(),
      sc.unit_work.as<uint32_t>(), cnt);
  k_units_fill<<<(int)((tt.nleaf + 255) / 256), 256, 0, s>>>(lv, tt.nleaf, tn, off, sc.unit_work.as<uint32_t>(), rows,
                                                             cnt, l.units.as<int4>(), l.multi.as<int4>());
  UVLM_LAUNCH_CHECK();
}

// Takes over what near_units_enqueue left at counters[UNIT_COUNTERS ..], read back by the caller, and
// reserves the partial sums.  False where the device has no room for them: the caller makes the units
// again with fewer rows (none at last), so that no call fails for the sake of its units.
bool near_units_set(Scratch &sc, const unsigned long long *h, Lists &l)
{
  l.n_interactions = (int64_t)h[NU_INTER];
  l.n_units        = (int64_t)h[NU_UNITS];
  l.n_rows         = (int64_t)h[NU_ROWS];
  l.n_multi        = (int64_t)h[NU_MULTI];
  l.wide           = h[NU_WIDE] != 0;
  if (l.n_rows > sc.near_rows) return false;
  try {
    sc.p2p_part.reserve(sizeof(double) * 12 * l.n_rows);
  } catch (const Error &e) {
    if (e.code != UVLM_ERR_NOMEM) throw;
    (void)hipGetLastError();
    return false;
  }
  return true;
}

// sensor_mode: 0 particles (u and J), 1 probes (u only), 2 adjoint (u and J, target sigma).
void p2p(hipStream_t s, Scratch &sc, const Tree &tt, const Tree &stree, const Lists &l, const double *tgt, int64_t tcap,
         const double *srcst, int64_t scap, double *out, int64_t ocap, int precision, int sensor_mode)
{
  if (tt.nleaf == 0) return;
  if (l.n_units < tt.nleaf) throw Error(UVLM_ERR_INTERNAL, "P2P without its units");
  double    *part  = sc.p2p_part.as<double>();
  const bool mixed = precision == UVLM_MIXED;
  auto       launch = [&](auto kern, int blk) {
    kern<<<(int)l.n_units, blk, 0, s>>>(l.units.as<int4>(), tt.leaves.as<int32_t>(), tt.body.as<int32_t>(),
                                        tt.nbody.as<int32_t>(), tt.cx.as<double>(), tt.cy.as<double>(),
                                        tt.cz.as<double>(), l.p2p_src.as<int32_t>(), stree.body.as<int32_t>(),
                                        stree.nbody.as<int32_t>(), tgt, tcap, srcst, scap, out, ocap, part);
  };
#define UVLM_P2P(MX, WJ, TS)                      \
  if (l.wide) launch(k_p2p<MX, WJ, TS, 256>, 256);   \
  else launch(k_p2p<MX, WJ, TS, 64>, 64)
  if (sensor_mode == 2) {
    if (mixed) UVLM_P2P(true, true, true);
    else UVLM_P2P(false, true, true);
  } else if (mixed && !sensor_mode) UVLM_P2P(true, true, false);
  else if (mixed) UVLM_P2P(true, false, false);
  else if (!sensor_mode) UVLM_P2P(false, true, false);
  else UVLM_P2P(false, false, false);
#undef UVLM_P2P
  UVLM_LAUNCH_CHECK();
  if (l.n_multi > 0) {
    auto reduce = [&](auto kern) {
      kern<<<(int)l.n_multi, 256, 0, s>>>(l.multi.as<int4>(), tt.leaves.as<int32_t>(), tt.body.as<int32_t>(),
                                          tt.nbody.as<int32_t>(), part, out, ocap);
    };
    if (sensor_mode != 1) reduce(k_p2p_reduce<true>);
    else reduce(k_p2p_reduce<false>);
    UVLM_LAUNCH_CHECK();
  }
}

// PSE (mode 0, adds prefix * sum to dadt) or Gaussian vorticity (mode 1, subtracts the sum
// from fields field..field+2) of the source tree at the target tree's leaves, over the P2P lists
// and their units.
void gauss_near(hipStream_t s, Scratch &sc, const Tree &tt, const Tree &stree, const Lists &l, const double *tgt,
                int64_t tcap, const double *srcst, int64_t scap, double *out, int64_t ocap, int mode, int field,
                double prefix)
{
  if (tt.nleaf == 0) return;
  if (l.n_units < tt.nleaf) throw Error(UVLM_ERR_INTERNAL, "Gaussian near field without its units");
  double        *part = sc.p2p_part.as<double>();
  const int32_t *lv = tt.leaves.as<int32_t>(), *tb = tt.body.as<int32_t>(), *tn = tt.nbody.as<int32_t>();
  auto           launch = [&](auto kern, int blk) {
    kern<<<(int)l.n_units, blk, 0, s>>>(l.units.as<int4>(), lv, tb, tn, l.p2p_src.as<int32_t>(),
                                        stree.body.as<int32_t>(), stree.nbody.as<int32_t>(), tgt, tcap, srcst, scap,
                                        out, ocap, field, prefix, part);
  };
  auto reduce = [&](auto kern) {
    if (l.n_multi > 0)
      kern<<<(int)l.n_multi, 256, 0, s>>>(l.multi.as<int4>(), lv, tb, tn, part, out, ocap, field, prefix);
  };
  if (mode == 0) {
    if (l.wide) launch(k_gauss<GAUSS_PSE, 256>, 256);
    else launch(k_gauss<GAUSS_PSE, 64>, 64);
    reduce(k_gauss_reduce<GAUSS_PSE>);
  } else {
    if (l.wide) launch(k_gauss<GAUSS_VORT, 256>, 256);
    else launch(k_gauss<GAUSS_VORT, 64>, 64);
    reduce(k_gauss_reduce<GAUSS_VORT>);
  }
  UVLM_LAUNCH_CHECK();
}

}  // namespace uvlm
