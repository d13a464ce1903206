// adjoint.hip -- vector-Jacobian product of the particle rates (velocity and stretching of one
// evaluation of FMMCalculator::calculate, src/fmmCalculator.hpp:420-467, cVPM), in FP64.
//
// With cotangents ubar_i (of u_i) and abar_i (of dadt_i) the objective is
//   S = sum_i ubar_i . u_i + Jbar_i : J_i,
//   Jbar_i = alpha_i abar_i^T (transposed stretching, dadt = J^T alpha) or abar_i alpha_i^T
//   (classic, dadt = J alpha),
// and the product returns xbar = dS/dx and alphabar = dS/dalpha for a frozen tree and lists:
//   alphabar_i = (J_i abar_i or J_i^T abar_i)                        the local stretching term
//              + sum_j [near] -W_ji + [far] curl(phi)(x_i) / (4 pi)  (phi below)
//   xbar_i     = sum_j [near, i target] dS_ij/dr - sum_j [near, i source] dS_ji/dr
//              + [far, i target] J_i^T ubar_i + Jbar_i : grad J_i
//              + [far, i source] (grad F)^T alpha_i,  F = curl(phi) / (4 pi).
// phi is the far field of the adjoint sources: vortices ubar_i and vortex dipoles Jbar_i at the
// particles (P2M of far.hip), carried by the same expansions along the TRANSPOSED M2L list:
// the total-degree truncation j + n <= P - 1 of M2L is the Taylor expansion of 1/|R + d| in
// d = (x_t - X_t) - (x_s - X_s), even in (R, d), so the adjoint of the far field is exactly the
// far field with targets and sources exchanged.
// Near pair (r = x_i - x_j, core sigma_j), with e the axial vector of Jbar_i:
//   S_ij = -alpha_j . W,   W = f1 (ubar_i x r + e) + f2 (Jbar_i r) x r,
//   dS_ij/dr = -[ f2 (alpha_j . (ubar_i x r + e)) r + f1 (alpha_j x ubar_i)
//                 + f3 (alpha_j . ((Jbar_i r) x r)) r + f2 Jbar_i^T (r x alpha_j)
//                 + f2 alpha_j x (Jbar_i r) ],
//   f1 = g / (4 pi R^3), f2 = (t2 / sigma^2 - 3 g / R^2) / (4 pi R^3),
//   f3 = (15 g / R^4 - t2 (5 + 2 s^2) / (sigma^2 R^2)) / (4 pi R^3),
// s^2 = R^2 / (2 sigma^2), t2 = (2/sqrt(pi)) s e^{-s^2}, g = erf(s) - t2 (the kernel of
// multipoleKernels.hpp:223-301 and its R^2 derivatives).
//
// Adjoint fields (SoA, `cap` doubles each): 0-2 ubar, 3-11 Jbar (row-major), 12-14 xbar,
// 15-17 alphabar.
#include "common.hpp"
#include "pair_kernel.hpp"

namespace uvlm {

namespace {

constexpr int WG = 64;

enum { A_UB = 0, A_JB = 3, A_XB = 12, A_AB = 15 };

template <class T> __device__ inline void cross(const T a[3], const T b[3], T o[3])
{
  o[0] = a[1] * b[2] - a[2] * b[1];
  o[1] = a[2] * b[0] - a[0] * b[2];
  o[2] = a[0] * b[1] - a[1] * b[0];
}

// G, G', G'' at x = R^2 q (pair_kernel.hpp).
__device__ __forceinline__ void pair_g(float r2, float q, float &G, float &Gp, float &Gpp)
{
  kernel_g<true>(r2 * q, G, Gp, Gpp);
}
__device__ __forceinline__ void pair_g(double r2, double q, double &G, double &Gp, double &Gpp)
{
  const double x = r2 * q;
  if (__double2hiint(x) < (int)X64_HI) {  // (x <= -0, of a core without a kernel, too: see core_q64)
    const double t = x - 0.5 * X64;
    double       g = c_g64[NG64 - 1], p = c_gp64[NG64 - 1], d = c_gpp64[NGPP64 - 1];
#pragma unroll
    for (int k = NG64 - 2; k >= 0; k--) {
      g = fma(g, t, c_g64[k]);
      p = fma(p, t, c_gp64[k]);
    }
#pragma unroll
    for (int k = NGPP64 - 2; k >= 0; k--) d = fma(d, t, c_gpp64[k]);
    G = g, Gp = p, Gpp = d;
  } else g64_far<true>(x, G, Gp, Gpp);
}
__device__ __forceinline__ float  fma_(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fma_(double a, double b, double c) { return fma(a, b, c); }

// Near-field adjoint, one workgroup per near-field unit of the (single) tree's list.  Like the
// forward P2P kernel, lanes = (own body) x (split s), the bodies of all listed leaves stream
// through LDS in chunks across leaf boundaries, and the splits and a leaf's units are added in a
// fixed order (deterministic, no atomics).
//  SIDE 0 (forward P2P list, own = target i):            xbar_i += sum_j dS_ij/dr
//  SIDE 1 (transposed list, own = source j): alphabar_j -= sum_i W_ij, xbar_j -= sum_i dS_ij/dr
// Sums over the pairs are arranged so that what belongs to the own body is applied once per
// chunk:
//  SIDE 0: sum_j dS_ij = -[X + F1 x ubar + Jbar^T V + A],  X = sum k r, F1 = sum f1 alpha_j,
//          V = sum f2 (r x alpha_j), A = sum f2 alpha_j x (Jbar r), k = f2 c1 + f3 c3;
//  SIDE 1: sum_i dS_ij = -[X + sum f2 Jbar_i^T (r x alpha) + alpha x sum (f1 ubar_i + f2 Jbar_i r)].
// MIXED: FP32 pair arithmetic on coordinates relative to the own leaf centre (formed in FP64
// while staging), FP32 partial sums of at most FLUSH entries a lane added into FP64 accumulators.
// Otherwise FP64 throughout.  Bound by VALU issue.  2.1e8 mixed pairs (260k blobs, P = 8,
// ncrit 64), against one wavefront per leaf and chunks of 64: SIDE 0 1.19 -> 0.60 ms, SIDE 1 1.48 ->
// 0.75 ms.
template <bool MIXED, int SIDE, int BLK>
__global__ __launch_bounds__(BLK) void k_p2p_adj(const int4 *__restrict__ units, const int32_t *__restrict__ leaves,
                                                 const int32_t *__restrict__ cbody, const int32_t *__restrict__ cnbody,
                                                 const double *__restrict__ ccx, const double *__restrict__ ccy,
                                                 const double *__restrict__ ccz, const int32_t *__restrict__ src,
                                                 const double *__restrict__ st, double *__restrict__ aux, int64_t cap,
                                                 double *__restrict__ part)
{
  using T = typename std::conditional<MIXED, float, double>::type;
  // staged per other body: SIDE 0: x, q, alpha, c1, c2, c3 (f_k = c_k G^(k-1));  SIDE 1: x, ubar, e, Jbar
  constexpr int NV = SIDE == 0 ? 10 : 18, NK = SIDE == 0 ? 3 : 6, CH = BLK;
  constexpr int SMEM = NV * CH * (int)sizeof(T) > NK * BLK * 8 ? NV * CH * (int)sizeof(T) : NK * BLK * 8;
  __shared__ __align__(16) unsigned char smem[SMEM];
  __shared__ int pref[SEG + 1], lb[SEG];
  T      *sv  = reinterpret_cast<T *>(smem);       // [CH][NV]
  double *red = reinterpret_cast<double *>(smem);  // [NK][BLK]
  const int4 un = units[blockIdx.x];
  const int  c = leaves[un.x], tb = cbody[c], nt = cnbody[c], q0 = un.y, q1 = un.z, prow = un.w, lane = threadIdx.x;
  const int    ntp = near_targets_per_pass<BLK>(nt), S = near_splits<BLK>(ntp), ti = lane % ntp, si = lane / ntp;
  const bool   lane_on = si < S;
  const double cxt = MIXED ? ccx[c] : 0.0, cyt = MIXED ? ccy[c] : 0.0, czt = MIXED ? ccz[c] : 0.0;
  for (int c0 = 0; c0 < nt; c0 += ntp) {
    const int     i      = c0 + ti;
    const int     jfirst = lane_on ? si : CH;  // lanes without a split skip the pair loops
    const int64_t bi     = tb + (lane_on && i < nt ? i : 0);
    const T       ro[3]  = {(T)(st[(F_X + 0) * cap + bi] - cxt), (T)(st[(F_X + 1) * cap + bi] - cyt),
                            (T)(st[(F_X + 2) * cap + bi] - czt)};
    // own quantities: SIDE 0 ubar, Jbar, e; SIDE 1 alpha, sigma and its kernel constants
    T      ub[3] = {0, 0, 0}, Jb[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, e[3] = {0, 0, 0}, al[3] = {0, 0, 0};
    double sgd = 1.0;
    if (SIDE == 0) {
      for (int d = 0; d < 3; d++) ub[d] = (T)aux[(A_UB + d) * cap + bi];
      for (int k = 0; k < 9; k++) Jb[k] = (T)aux[(A_JB + k) * cap + bi];
      e[0] = Jb[5] - Jb[7], e[1] = Jb[6] - Jb[2], e[2] = Jb[1] - Jb[3];
    } else {
      for (int d = 0; d < 3; d++) al[d] = (T)st[(F_A + d) * cap + bi];
      sgd = st[F_SIG * cap + bi];
    }
    const double oqd = MIXED ? 0.5 / (sgd * sgd) : core_q64(sgd), oc1 = pow32(oqd) * INV_4PI;
    const T      o_q = (T)oqd, o_c1 = (T)oc1, o_c2 = (T)(2.0 * oqd * oc1), o_c3 = (T)(4.0 * oqd * oqd * oc1);
    double       ax[3] = {0, 0, 0}, aa[3] = {0, 0, 0};
    for (int g0 = q0; g0 < q1; g0 += SEG) {
      const int nseg = min(SEG, q1 - g0);
      __syncthreads();
      for (int k = lane; k < nseg; k += BLK) {
        const int sl = src[g0 + k];
        lb[k]        = cbody[sl];
        pref[k]      = cnbody[sl];
      }
      __syncthreads();
      if (lane < 64) lds_prefix(pref, pref, nseg);
      __syncthreads();
      const int total = pref[nseg];
      for (int j0 = 0; j0 < total; j0 += CH) {
        const int cnt = min(CH, total - j0);
        if (lane < cnt) {
          const int64_t bj = list_body(pref, lb, nseg, j0 + lane);
          T            *v  = sv + NV * lane;
          v[0] = (T)(st[(F_X + 0) * cap + bj] - cxt);
          v[1] = (T)(st[(F_X + 1) * cap + bj] - cyt);
          v[2] = (T)(st[(F_X + 2) * cap + bj] - czt);
          if (SIDE == 0) {
            const double sg = st[F_SIG * cap + bj], qq = MIXED ? 0.5 / (sg * sg) : core_q64(sg);
            v[3] = (T)qq;
            for (int d = 0; d < 3; d++) v[4 + d] = (T)st[(F_A + d) * cap + bj];
            const double c1 = pow32(qq) * INV_4PI;
            v[7] = (T)c1, v[8] = (T)(2.0 * qq * c1), v[9] = (T)(4.0 * qq * qq * c1);
          } else {
            double Jd[9];
            for (int d = 0; d < 3; d++) v[3 + d] = (T)aux[(A_UB + d) * cap + bj];
            for (int k = 0; k < 9; k++) Jd[k] = aux[(A_JB + k) * cap + bj];
            v[6] = (T)(Jd[5] - Jd[7]), v[7] = (T)(Jd[6] - Jd[2]), v[8] = (T)(Jd[1] - Jd[3]);
            for (int k = 0; k < 9; k++) v[9 + k] = (T)Jd[k];
          }
        }
        __syncthreads();
        // SIDE 0: X, F1, V, A;  SIDE 1: X, JV, UQ, WA
        constexpr int FLUSH = 64;
        for (int k0 = jfirst; k0 < cnt; k0 += FLUSH * S) {
          T p0[3] = {0, 0, 0}, p1[3] = {0, 0, 0}, p2[3] = {0, 0, 0}, p3[3] = {0, 0, 0};
          const int kend = min(cnt, k0 + FLUSH * S);
          for (int j = k0; j < kend; j += S) {
            const T *v    = sv + NV * j;
            const T  sgn1 = SIDE == 0 ? (T)1 : (T)-1;
            const T  r[3] = {sgn1 * (ro[0] - v[0]), sgn1 * (ro[1] - v[1]), sgn1 * (ro[2] - v[2])};
            const T  r2   = r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
            const T  q    = SIDE == 0 ? v[3] : o_q;
            T        G, Gp, Gpp;
            pair_g(r2, q, G, Gp, Gpp);
            // coincident pairs are skipped (multipoleKernels.hpp:242): every term but the f1 ones
            // carries r, so zeroing f1 is enough
            const T f1 = r2 == (T)0 ? (T)0 : G * (SIDE == 0 ? v[7] : o_c1);
            const T f2 = Gp * (SIDE == 0 ? v[8] : o_c2), f3 = Gpp * (SIDE == 0 ? v[9] : o_c3);
            if (SIDE == 0) {
              const T aj[3] = {v[4], v[5], v[6]};
              T       w[3], Jr[3], aJ[3];
              cross(r, aj, w);
              for (int d = 0; d < 3; d++) Jr[d] = Jb[3 * d] * r[0] + Jb[3 * d + 1] * r[1] + Jb[3 * d + 2] * r[2];
              cross(aj, Jr, aJ);
              const T cc1 = ub[0] * w[0] + ub[1] * w[1] + ub[2] * w[2] + aj[0] * e[0] + aj[1] * e[1] + aj[2] * e[2];
              const T cc3 = Jr[0] * w[0] + Jr[1] * w[1] + Jr[2] * w[2];
              const T k   = f2 * cc1 + f3 * cc3;
              for (int d = 0; d < 3; d++) {
                p0[d] = fma_(k, r[d], p0[d]);
                p1[d] = fma_(f1, aj[d], p1[d]);
                p2[d] = fma_(f2, w[d], p2[d]);
                p3[d] = fma_(f2, aJ[d], p3[d]);
              }
            } else {
              const T *bu = v + 3, *be = v + 6, *bJ = v + 9;
              T        uxr[3], Jr[3], Jrxr[3], w[3];
              cross(bu, r, uxr);
              for (int d = 0; d < 3; d++) Jr[d] = bJ[3 * d] * r[0] + bJ[3 * d + 1] * r[1] + bJ[3 * d + 2] * r[2];
              cross(Jr, r, Jrxr);
              cross(r, al, w);
              T cc1 = 0, cc3 = 0;
              for (int d = 0; d < 3; d++) {
                cc1 = fma_(al[d], uxr[d] + be[d], cc1);
                cc3 = fma_(al[d], Jrxr[d], cc3);
              }
              const T k = f2 * cc1 + f3 * cc3;
              for (int d = 0; d < 3; d++) {
                const T JTw = bJ[d] * w[0] + bJ[3 + d] * w[1] + bJ[6 + d] * w[2];
                p0[d]       = fma_(k, r[d], p0[d]);
                p1[d]       = fma_(f2, JTw, p1[d]);
                p2[d]       = fma_(f1, bu[d], fma_(f2, Jr[d], p2[d]));
                p3[d]       = fma_(f1, uxr[d] + be[d], fma_(f2, Jrxr[d], p3[d]));
              }
            }
          }
          if (SIDE == 0) {
            // sum dS = -[X + F1 x ubar + Jbar^T V + A]
            T fxu[3];
            cross(p1, ub, fxu);
            for (int d = 0; d < 3; d++) {
              const T JTV = Jb[d] * p2[0] + Jb[3 + d] * p2[1] + Jb[6 + d] * p2[2];
              ax[d] -= (double)(p0[d] + fxu[d] + JTV + p3[d]);
            }
          } else {
            // xbar_j -= sum dS = X + JV + alpha x UQ;  alphabar_j -= sum W
            T axq[3];
            cross(al, p2, axq);
            for (int d = 0; d < 3; d++) {
              ax[d] += (double)(p0[d] + p1[d] + axq[d]);
              aa[d] -= (double)p3[d];
            }
          }
        }
        __syncthreads();
      }
    }
    // the splits (lanes t + q * ntp) in split order; lanes then take (field, body)
    const int np = min(ntp, nt - c0);
    __syncthreads();
    for (int d = 0; d < 3; d++) {
      red[d * BLK + lane] = ax[d];
      if (SIDE == 1) red[(3 + d) * BLK + lane] = aa[d];
    }
    __syncthreads();
    for (int o = lane; o < NK * np; o += BLK) {
      const int k = o / np, tt = o - k * np;
      double    v = red[k * BLK + tt];
      for (int q = 1; q < S; q++) v += red[k * BLK + tt + q * ntp];
      if (prow >= 0) part[(int64_t)prow * 12 + (int64_t)k * nt + c0 + tt] = v;
      else aux[(A_XB + k) * cap + tb + c0 + tt] += v;  // A_AB = A_XB + 3
    }
  }
}
static_assert(A_AB == A_XB + 3, "xbar and alphabar fields are consecutive");

// Sums of the leaves cut into several units, units in order.
template <int SIDE>
__global__ __launch_bounds__(256) void k_p2p_adj_reduce(const int4 *__restrict__ multi,
                                                        const int32_t *__restrict__ leaves,
                                                        const int32_t *__restrict__ cbody,
                                                        const int32_t *__restrict__ cnbody,
                                                        const double *__restrict__ part, double *__restrict__ aux,
                                                        int64_t cap)
{
  const int4    m = multi[blockIdx.x];
  const int     c = leaves[m.x], tb = cbody[c], nt = cnbody[c];
  const double *p = part + (int64_t)m.y * 12;
  for (int o = threadIdx.x; o < (SIDE == 0 ? 3 : 6) * nt; o += 256) {
    const int k = o / nt;
    double    v = 0.0;
#pragma unroll 4
    for (int u = 0; u < m.z; u++) v += p[(int64_t)u * 12 * nt + o];
    aux[(A_XB + k) * cap + tb + (o - k * nt)] += v;
  }
}

// Jbar from alpha and abar (abar uploaded into the alphabar fields), the local stretching term
// of alphabar (J abar or J^T abar with the forward J), xbar cleared.
__global__ void k_vjp_setup(int64_t N, const double *__restrict__ st, double *__restrict__ aux, int64_t cap,
                            int classic)
{
  const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (i >= N) return;
  double al[3], ab[3], J[9];
  for (int d = 0; d < 3; d++) {
    al[d] = st[(F_A + d) * cap + i];
    ab[d] = aux[(A_AB + d) * cap + i];
  }
  for (int k = 0; k < 9; k++) J[k] = st[(F_J + k) * cap + i];
  for (int a = 0; a < 3; a++)
    for (int b = 0; b < 3; b++) aux[(A_JB + 3 * a + b) * cap + i] = classic ? ab[a] * al[b] : al[a] * ab[b];
  for (int a = 0; a < 3; a++) {
    double v = 0.0;
    for (int b = 0; b < 3; b++) v += classic ? J[3 * b + a] * ab[b] : J[3 * a + b] * ab[b];
    aux[(A_AB + a) * cap + i] = v;
    aux[(A_XB + a) * cap + i] = 0.0;
  }
}

// Far source-side terms from the adjoint L2P (ast: velocity = F, dadt = (grad F)^T alpha).
__global__ void k_vjp_finish(int64_t N, const double *__restrict__ ast, double *__restrict__ aux, int64_t cap)
{
  const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (i >= N) return;
  for (int d = 0; d < 3; d++) {
    aux[(A_XB + d) * cap + i] += ast[(F_DADT + d) * cap + i];
    aux[(A_AB + d) * cap + i] += ast[(F_U + d) * cap + i];
  }
}

// Cotangents of the state (X, alpha) live in the original body order: 6 SoA fields of `ccap`
// doubles (0-2 position, 3-5 strength).  orig[p] is the original index of device body p.
__global__ void k_cot_gather(int64_t N, const int32_t *__restrict__ orig, const double *__restrict__ cot,
                             int64_t ccap, double *__restrict__ aux, int64_t cap)
{
  const int64_t p = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (p >= N) return;
  const int64_t o = orig[p];
  for (int d = 0; d < 3; d++) {
    aux[(A_UB + d) * cap + p] = cot[d * ccap + o];
    aux[(A_AB + d) * cap + p] = cot[(3 + d) * ccap + o];
  }
}

__global__ void k_cot_scatter(int64_t N, const int32_t *__restrict__ orig, const double *__restrict__ aux,
                              int64_t cap, double *__restrict__ cot, int64_t ccap)
{
  const int64_t p = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (p >= N) return;
  const int64_t o = orig[p];
  for (int d = 0; d < 3; d++) {
    cot[d * ccap + o]       = aux[(A_XB + d) * cap + p];
    cot[(3 + d) * ccap + o] = aux[(A_AB + d) * cap + p];
  }
}

__global__ void k_state_to_orig(int64_t N, const int32_t *__restrict__ orig, const double *__restrict__ st,
                                int64_t cap, double *__restrict__ dst)
{
  const int64_t p = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (p >= N) return;
  const int64_t o = orig[p];
  for (int f = 0; f < 6; f++) dst[f * N + o] = st[(F_X + f) * cap + p];
  dst[6 * N + o] = st[F_SIG * cap + p];
}

struct LinTerms {
  const double *p[6];
  double        c[6];
  int           n;
};

__global__ void k_lincomb(int64_t n, double *__restrict__ out, LinTerms t)
{
  const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (i >= n) return;
  double v = 0.0;
  for (int k = 0; k < t.n; k++) v += t.c[k] * t.p[k][i];
  out[i] = v;
}

}  // namespace

void cot_gather(hipStream_t s, int64_t N, const int32_t *orig, const double *cot, int64_t ccap, double *aux,
                int64_t cap)
{
  if (N <= 0) return;
  k_cot_gather<<<(int)((N + 255) / 256), 256, 0, s>>>(N, orig, cot, ccap, aux, cap);
  UVLM_LAUNCH_CHECK();
}

void cot_scatter(hipStream_t s, int64_t N, const int32_t *orig, const double *aux, int64_t cap, double *cot,
                 int64_t ccap)
{
  if (N <= 0) return;
  k_cot_scatter<<<(int)((N + 255) / 256), 256, 0, s>>>(N, orig, aux, cap, cot, ccap);
  UVLM_LAUNCH_CHECK();
}

void state_to_orig(hipStream_t s, int64_t N, const int32_t *orig, const double *st, int64_t cap, double *dst)
{
  if (N <= 0) return;
  k_state_to_orig<<<(int)((N + 255) / 256), 256, 0, s>>>(N, orig, st, cap, dst);
  UVLM_LAUNCH_CHECK();
}

void lincomb(hipStream_t s, int64_t n, double *out, int nterms, const double *const *p, const double *c)
{
  if (n <= 0) return;
  if (nterms > 6) throw Error(UVLM_ERR_INTERNAL, "lincomb: more than 6 terms");
  LinTerms t{};
  t.n = nterms;
  for (int k = 0; k < nterms; k++) {
    t.p[k] = p[k];
    t.c[k] = c[k];
  }
  k_lincomb<<<(int)((n + 255) / 256), 256, 0, s>>>(n, out, t);
  UVLM_LAUNCH_CHECK();
}

void vjp_setup(hipStream_t s, int64_t N, const double *st, double *aux, int64_t cap, int classic)
{
  if (N <= 0) return;
  k_vjp_setup<<<(int)((N + 255) / 256), 256, 0, s>>>(N, st, aux, cap, classic);
  UVLM_LAUNCH_CHECK();
}

void vjp_finish(hipStream_t s, int64_t N, const double *ast, double *aux, int64_t cap)
{
  if (N <= 0) return;
  k_vjp_finish<<<(int)((N + 255) / 256), 256, 0, s>>>(N, ast, aux, cap);
  UVLM_LAUNCH_CHECK();
}

// Cotangent of the sources' core sizes, sbar_j = dS/dsigma_j (device order of the sources), of
// S = sum over the near (P2P) pairs of ubar_i . u_i + Jbar_i : J_i: only the near field depends
// on sigma (the far field applies the singular kernel).  Per pair, r = x_i - x_j and the kernel of
// sigma_j, S_ij = -alpha_j . (f1 (ubar_i x r + e_i) + f2 (Jbar_i r) x r), e the axial vector of
// Jbar, so dS_ij/dsigma_j = -alpha_j . (f1s (ubar_i x r + e_i) + f2s (Jbar_i r) x r) with
// f1s = df1/dsigma = -2 s^2 t2 / (sigma 4 pi R^3), f2s = df2/dsigma = 2 s^2 t2 / (sigma^3 4 pi R^3),
// s^2 = R^2 / (2 sigma^2), t2 = 2 s e^{-s^2} / sqrt(pi).  FP64.  One wavefront per source leaf,
// lanes over its bodies; `off`/`ent` is CSR by source cell with target cells as entries (the
// P2P list transposed); the target bodies pass through LDS, 64 at a time, in list order.
template <bool WITH_JB>
__global__ __launch_bounds__(WG) void k_sigma_bar(const int32_t *__restrict__ leaves, int64_t nleaf,
                                                  const int32_t *__restrict__ sbody, const int32_t *__restrict__ snb,
                                                  const int32_t *__restrict__ off, const int32_t *__restrict__ ent,
                                                  const int32_t *__restrict__ tbody, const int32_t *__restrict__ tnb,
                                                  const double *__restrict__ tx, int64_t tcap,
                                                  const double *__restrict__ tcot, int64_t ccap,
                                                  const double *__restrict__ sst, int64_t scap,
                                                  double *__restrict__ sbar)
{
  __shared__ double sh[15][WG];
  const int64_t w = blockIdx.x;
  if (w >= nleaf) return;
  const int lane = threadIdx.x;
  const int sl = leaves[w], sb0 = sbody[sl], ns = snb[sl];
  for (int p0 = 0; p0 < ns; p0 += WG) {
    const int  j  = sb0 + p0 + lane;
    const bool ok = p0 + lane < ns;
    double     xj[3] = {0, 0, 0}, aj[3] = {0, 0, 0}, sg = 1.0;
    if (ok) {
      for (int d = 0; d < 3; d++) {
        xj[d] = sst[(F_X + d) * scap + j];
        aj[d] = sst[(F_A + d) * scap + j];
      }
      sg = sst[F_SIG * scap + j];
    }
    const double S2 = sg * sg;
    double       acc = 0.0;
    for (int q = off[sl]; q < off[sl + 1]; q++) {
      const int t = ent[q], tb0 = tbody[t], nt = tnb[t];
      for (int c0 = 0; c0 < nt; c0 += WG) {
        const int cnt = min(WG, nt - c0);
        __syncthreads();
        if (lane < cnt) {
          const int64_t i = tb0 + c0 + lane;
          for (int d = 0; d < 3; d++) {
            sh[d][lane]     = tx[(F_X + d) * tcap + i];
            sh[3 + d][lane] = tcot[d * ccap + i];
          }
          if (WITH_JB)
            for (int k = 0; k < 9; k++) sh[6 + k][lane] = tcot[(3 + k) * ccap + i];
        }
        __syncthreads();
        if (!ok) continue;
        for (int e = 0; e < cnt; e++) {
          const double r[3] = {sh[0][e] - xj[0], sh[1][e] - xj[1], sh[2][e] - xj[2]};
          const double R2   = r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
          if (R2 == 0.0) continue;
          const double s2 = R2 / S2 * 0.5, t2 = 2.0 * INV_SQRTPI * sqrt(s2) * exp(-s2);
          const double q4 = 0.25 * INV_PI / (R2 * sqrt(R2));
          const double f1s = -2.0 * s2 * t2 * q4 / sg, f2s = 2.0 * s2 * t2 * q4 / (S2 * sg);
          const double ub[3] = {sh[3][e], sh[4][e], sh[5][e]};
          double       W[3]  = {ub[1] * r[2] - ub[2] * r[1], ub[2] * r[0] - ub[0] * r[2], ub[0] * r[1] - ub[1] * r[0]};
          for (int d = 0; d < 3; d++) W[d] *= f1s;
          if (WITH_JB) {
            const double *M = &sh[6][0];
            auto          Jb = [&](int a, int b) { return M[(3 * a + b) * WG + e]; };
            const double  ea[3] = {Jb(1, 2) - Jb(2, 1), Jb(2, 0) - Jb(0, 2), Jb(0, 1) - Jb(1, 0)};
            double        Jr[3];
            for (int a = 0; a < 3; a++) Jr[a] = Jb(a, 0) * r[0] + Jb(a, 1) * r[1] + Jb(a, 2) * r[2];
            const double Jrxr[3] = {Jr[1] * r[2] - Jr[2] * r[1], Jr[2] * r[0] - Jr[0] * r[2],
                                    Jr[0] * r[1] - Jr[1] * r[0]};
            for (int d = 0; d < 3; d++) W[d] += f1s * ea[d] + f2s * Jrxr[d];
          }
          acc -= aj[0] * W[0] + aj[1] * W[1] + aj[2] * W[2];
        }
      }
    }
    if (ok) sbar[j] = acc;
  }
}

__global__ void k_add_to_orig(int64_t N, const int32_t *__restrict__ orig, const double *__restrict__ src,
                              double *__restrict__ dst)
{
  const int64_t p = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (p >= N) return;
  dst[orig[p]] += src[p];
}

void add_to_orig(hipStream_t s, int64_t N, const int32_t *orig, const double *src, double *dst)
{
  if (N <= 0) return;
  k_add_to_orig<<<(int)((N + 255) / 256), 256, 0, s>>>(N, orig, src, dst);
  UVLM_LAUNCH_CHECK();
}

void sigma_bar(hipStream_t s, const Tree &stree, const Tree &ttree, const Lists &tl, const double *tx, int64_t tcap,
               const double *tcot, int64_t ccap, bool with_jbar, const double *sst, int64_t scap, double *sbar)
{
  if (stree.nleaf == 0) return;
  const int32_t *lv = stree.leaves.as<int32_t>(), *sb = stree.body.as<int32_t>(), *sn = stree.nbody.as<int32_t>();
  const int32_t *off = tl.p2p_off.as<int32_t>(), *ent = tl.p2p_src.as<int32_t>();
  const int32_t *tb = ttree.body.as<int32_t>(), *tn = ttree.nbody.as<int32_t>();
  const int      nb = (int)stree.nleaf;
  if (with_jbar)
    k_sigma_bar<true><<<nb, WG, 0, s>>>(lv, stree.nleaf, sb, sn, off, ent, tb, tn, tx, tcap, tcot, ccap, sst, scap, sbar);
  else
    k_sigma_bar<false><<<nb, WG, 0, s>>>(lv, stree.nleaf, sb, sn, off, ent, tb, tn, tx, tcap, tcot, ccap, sst, scap,
                                         sbar);
  UVLM_LAUNCH_CHECK();
}

void p2p_adj(hipStream_t s, Scratch &sc, const Tree &t, const Lists &l, int side, int mixed, const double *st,
             double *aux, int64_t cap)
{
  if (t.nleaf == 0) return;
  if (l.n_units < t.nleaf) throw Error(UVLM_ERR_INTERNAL, "near-field adjoint without its units");
  double        *part = sc.p2p_part.as<double>();
  const int32_t *lv = t.leaves.as<int32_t>(), *cb = t.body.as<int32_t>(), *cn = t.nbody.as<int32_t>();
  auto           launch = [&](auto kern, int blk) {
    kern<<<(int)l.n_units, blk, 0, s>>>(l.units.as<int4>(), lv, cb, cn, t.cx.as<double>(), t.cy.as<double>(),
                                        t.cz.as<double>(), l.p2p_src.as<int32_t>(), st, aux, cap, part);
  };
#define UVLM_ADJ(MX, SD)                          \
  if (l.wide) launch(k_p2p_adj<MX, SD, 256>, 256); \
  else launch(k_p2p_adj<MX, SD, 64>, 64)
  if (mixed) {
    if (side == 0) UVLM_ADJ(true, 0);
    else UVLM_ADJ(true, 1);
  } else {
    if (side == 0) UVLM_ADJ(false, 0);
    else UVLM_ADJ(false, 1);
  }
#undef UVLM_ADJ
  if (l.n_multi > 0) {
    auto reduce = [&](auto kern) {
      kern<<<(int)l.n_multi, 256, 0, s>>>(l.multi.as<int4>(), lv, cb, cn, part, aux, cap);
    };
    if (side == 0) reduce(k_p2p_adj_reduce<0>);
    else reduce(k_p2p_adj_reduce<1>);
  }
  UVLM_LAUNCH_CHECK();
}

}  // namespace uvlm
