// pair_kernel.hpp -- FP32 evaluation of the regularised Biot-Savart kernel factor and its
// derivatives (shared by the near-field kernels and their adjoint), and the LDS prefix sum
// the near-field kernels use to stream the bodies of several leaves in full chunks.
//
// With s = R / (sqrt(2) sigma), x = s^2, g = erf(s) - t2, t2 = (2/sqrt(pi)) s e^{-s^2}
// (multipoleKernels.hpp:243-283), the pair factors are functions of G(x) = g / s^3:
//   f1 = g / (4 pi R^3)   = G(x)   q^{3/2} / (4 pi),
//   f2 = 2 df1/dR^2       = 2 G'(x)  q^{5/2} / (4 pi),
//   f3 = 2 df2/dR^2       = 4 G''(x) q^{7/2} / (4 pi),      q = 1 / (2 sigma^2),
// because 2 s^2 t2 - 3 g = s g'(s) - 3 g = 2 s^5 G'(x), and
//   G(x) = (2/sqrt(pi)) sum_{i>=0} (-1)^i 2(i+1) / ((2i+3) (i+1)!) x^i.
// For x < 2, G is approximated on [0, 2] by its degree-9 Chebyshev interpolant (kernel_g, which
// also needs G''; the forward kernels interpolate G and G' separately, c_gnear and c_gpnear
// below) (interpolation at the Chebyshev nodes of [0, 2], re-expanded in powers of t = x - 1),
// with no cancellation between erf and t2: max error 8e-11 (G), 5e-9 (G') and 7.6e-8 (G'',
// |G''| <= 0.33) in exact arithmetic, 1.4e-7 and 1.1e-7 (G, G') when evaluated by Horner in FP32.
// For x >= 2 the hardware rsq/exp2 and a short polynomial: with w = x^{-1/2} = 1/s, e = e^{-x},
//   g = erf(s) - (2/sqrt(pi)) s e = 1 - e (erfcx(s) + (2/sqrt(pi)) s),
//   G = g w^3,   G' = w^2 ((2/sqrt(pi)) e - (3/2) G),
//   G'' = -(2/sqrt(pi)) e (w^2 + w^4) - (3/2) w^2 (G' - G w^2)
// (from G' = (2/sqrt(pi)) s e x^{-3/2} - (3/2) G / x), where erfcx(s) = e^{s^2} erfc(s) is a
// degree-7 least-squares polynomial in w - 0.4647 on w in [1/4.5, 1/sqrt(2)] (max error
// 1e-8; beyond s = 4.5 the factor e < 2e-9 makes it irrelevant, so w is clamped there).
// In FP32 this form is as accurate as erff/expf (4.3e-7 on G, 8.1e-7 on G') for about a
// third of the instructions.
#pragma once
#include <hip/hip_runtime.h>

namespace uvlm {
namespace {

// Chebyshev interpolant of G on x in [0, 2], coefficients of t^i, t = x - 1.
constexpr int   NPOLY              = 10;
constexpr float XPOLY              = 2.0f;
__constant__ float c_gpoly[NPOLY] = {4.27593295550599495e-01f,  -2.26282445882890593e-01f, 7.52993075578484716e-02f,
                                     -1.86646103035026413e-02f, 3.70154966273965411e-03f,  -6.12467145832412121e-04f,
                                     8.69427232794296300e-05f,  -1.08135023163257920e-05f, 1.22398144588401693e-06f,
                                     -1.21730778572683114e-07f};

// The forward near-field kernels need G and G' only: each has its own degree-7 interpolant at
// the Chebyshev nodes of [0, 2] (coefficients of t^i, t = x - 1), accurate to 1.1e-8 (G) and
// 9.5e-9 (G') in exact arithmetic and to 7.3e-8 and 4.3e-8 by fused Horner in FP32.  Two chains
// of 7 multiply-adds, independent of each other, instead of one degree-8 polynomial and its
// derivative (15 multiply-adds, the derivative's chain waiting on the value's).
constexpr int   NNEAR              = 8;
__constant__ float c_gnear[NNEAR]  = {4.27593286009723905e-01f,  -2.26282444927409232e-01f, 7.52996131662352769e-02f,
                                      -1.86646407540406734e-02f, 3.70002071831887491e-03f,  -6.12314968091220990e-04f,
                                      8.93899977314482896e-05f,  -1.10569638636093259e-05f};
__constant__ float c_gpnear[NNEAR] = {-2.26282437333498510e-01f, 1.50598616404860219e-01f,  -5.59941046870113882e-02f,
                                      1.48061917699502943e-02f,  -3.06096641491382382e-03f, 5.21663223968849010e-04f,
                                      -7.78856703251840088e-05f, 9.79185156779749377e-06f};

// erfcx(1/w) ~ sum_k c_far[k] (w - FAR_WC)^k, w in [FAR_WMIN, 1/sqrt(2)].
constexpr int   NFAR     = 8;
constexpr float FAR_WC   = 0.46466450170438484f;
constexpr float FAR_WMIN = 0.2222222222222222f;
__constant__ float c_far[NFAR] = {2.400683016e-01f,  4.403707087e-01f, -1.874301285e-01f, 1.258202083e-02f,
                                  8.160093427e-02f, -1.016800180e-01f, 5.416155234e-02f,  2.011496387e-02f};

// G, G' and (D2) G'' at x = xq >= 0.
template <bool D2>
__device__ __forceinline__ void kernel_g(float xq, float &G, float &Gp, float &Gpp)
{
  if (xq < XPOLY) {
    const float tq = xq - 1.0f;
    float       g = c_gpoly[NPOLY - 1], gp = 0.f, gpp = 0.f;
#pragma unroll
    for (int k = NPOLY - 2; k >= 0; k--) {
      if (D2) gpp = fmaf(gpp, tq, gp);
      gp = fmaf(gp, tq, g);
      g  = fmaf(g, tq, c_gpoly[k]);
    }
    G   = g;
    Gp  = gp;
    Gpp = 2.0f * gpp;
  } else {
    const float w = __builtin_amdgcn_rsqf(xq);
    const float e = __builtin_amdgcn_exp2f(xq * -1.4426950408889634f);
    const float t = fmaxf(w, FAR_WMIN) - FAR_WC;
    float       p = c_far[NFAR - 1];
#pragma unroll
    for (int k = NFAR - 2; k >= 0; k--) p = fmaf(p, t, c_far[k]);
    const float g  = fmaf(-e, fmaf(1.1283791670955126f, xq * w, p), 1.0f);
    const float w2 = w * w;
    G              = g * w2 * w;
    Gp             = w2 * fmaf(1.1283791670955126f, e, -1.5f * G);
    if (D2) Gpp = -1.1283791670955126f * e * fmaf(w2, w2, w2) - 1.5f * w2 * fmaf(-G, w2, Gp);
  }
}

// G, G' at t0 = x0 - 1 and t1 = x1 - 1 (x < XPOLY) by the degree-7 interpolants: four
// independent Horner chains, each started after its first step.
__device__ __forceinline__ void g_near(float t0, float t1, float &G0, float &Gp0, float &G1, float &Gp1)
{
  float g0 = fmaf(c_gnear[NNEAR - 1], t0, c_gnear[NNEAR - 2]), g1 = fmaf(c_gnear[NNEAR - 1], t1, c_gnear[NNEAR - 2]);
  float p0 = fmaf(c_gpnear[NNEAR - 1], t0, c_gpnear[NNEAR - 2]), p1 = fmaf(c_gpnear[NNEAR - 1], t1, c_gpnear[NNEAR - 2]);
#pragma unroll
  for (int k = NNEAR - 3; k >= 0; k--) {
    g0 = fmaf(g0, t0, c_gnear[k]);
    g1 = fmaf(g1, t1, c_gnear[k]);
    p0 = fmaf(p0, t0, c_gpnear[k]);
    p1 = fmaf(p1, t1, c_gpnear[k]);
  }
  G0 = g0, Gp0 = p0, G1 = g1, Gp1 = p1;
}

// G, G' at x >= XPOLY from rsq/exp2 and the erfcx polynomial (the x >= XPOLY branch of kernel_g).
__device__ __forceinline__ void g_far(float xq, float &G, float &Gp)
{
  const float w = __builtin_amdgcn_rsqf(xq);
  const float e = __builtin_amdgcn_exp2f(xq * -1.4426950408889634f);
  const float t = fmaxf(w, FAR_WMIN) - FAR_WC;
  float       p = c_far[NFAR - 1];
#pragma unroll
  for (int k = NFAR - 2; k >= 0; k--) p = fmaf(p, t, c_far[k]);
  const float g  = fmaf(-e, fmaf(1.1283791670955126f, xq * w, p), 1.0f);
  const float w2 = w * w;
  G              = g * w2 * w;
  Gp             = w2 * fmaf(1.1283791670955126f, e, -1.5f * G);
}

// ---- FP64 pair factors --------------------------------------------------------------------
// The FP64 near field used the reference formula with the library's erf, exp, sqrt and three
// divisions: about 250 instructions a pair (11.0 ms for 1.54e9 pairs of the 1M two rings).
// Here G and G' (and G'' for the adjoint) come from polynomials too:
//  * x < X64 = 3: degree-16 interpolants of G and G' (17 for G'') at the Chebyshev nodes of
//    [0, 3] in t = x - 3/2: relative error 3.5e-18, 8.4e-18 and 5.7e-19 in exact arithmetic and
//    1.7e-16, 2.2e-16, 2.2e-16 by fused Horner.  Unlike erf - t2 there is no cancellation at
//    small x (the formula loses a factor 1/x on f1 and 1/x^2 on f2).  3 rather than 2 (degree 14)
//    costs 4 multiply-adds a pair and keeps more waves off the far form; 4 needs degree 18.
//  * x >= 3: g = 1 - e^{-x} (erfcx(s) + (2/sqrt(pi)) s) as in FP32, with rsq refined by one cubic
//    step, e^r on |r| <= ln 2 / 2 by its degree-11 interpolant at the Chebyshev nodes there (c_exp64,
//    computed in 60 digits as the others), and erfcx as a degree-11 minimax polynomial in
//    w = 1/s whose error weighted by e^{-x} is 1.2e-17.  From x = FAR64 = 44 on, e^{-x} no longer
//    shows in G or G' and a wave all of whose lanes are there skips it.
constexpr double X64 = 3.0, FAR64 = 44.0;
constexpr unsigned X64_HI = 0x40080000u;  // high word of X64: x < X64 where the high word is below
constexpr int NG64 = 17, NGPP64 = 18, NFAR64 = 12, NEXP64 = 12;
constexpr double FAR64_WC = 0.3640529707392538, FAR64_WMIN = 0.15075567228888181;
constexpr double TWO_SQRTPI = 1.1283791670955126;
__constant__ double c_g64[17] = {
    3.31157308998109245e-01, -1.63307026156660179e-01, 5.21640470431589676e-02, -1.25969894488822884e-02,
    2.45398030160123067e-03, -4.00833197494527367e-04, 5.63652498002339511e-05, -6.95726516926421291e-06,
    7.65109382981209354e-07, -7.58599198635941649e-08, 6.84690821463335333e-09, -5.67087542187630871e-10,
    4.33916973335413845e-11, -3.08354343847775088e-12, 2.04760655365041072e-13, -1.31590474790122235e-14,
    7.69092086651117093e-16};
__constant__ double c_gp64[17] = {
    -1.63307026156660207e-01, 1.04328094086317935e-01, -3.77909683466464003e-02, 9.81592120640503718e-03,
    -2.00416598747744749e-03, 3.38191498800797814e-04, -4.87008561660276932e-05, 6.12087506526053526e-06,
    -6.82739314636161485e-07, 6.84690804739502330e-08, -6.23792611506433268e-09, 5.20701422245581422e-10,
    -4.01069139650919117e-11, 2.86631274157453670e-12, -1.91274669263023203e-13, 1.23481991649719220e-14,
    -7.24413669201184165e-16};
__constant__ double c_gpp64[18] = {
    1.04328094086317935e-01, -7.55819366932928005e-02, 2.94477636192146709e-02, -8.01666394990975875e-03,
    1.69095749400854705e-03, -2.92205136996453215e-04, 4.28461254389931391e-05, -5.46191451601966715e-06,
    6.16221758233975666e-07, -6.23792631318532978e-08, 5.72768074901313056e-09, -4.81280969224836532e-10,
    3.72818068782074733e-11, -2.67896141427953826e-12, 1.79437434662867233e-13, -1.12666500869749876e-14,
    6.85754757690162003e-16, -3.81177028769169991e-17};
__constant__ double c_far64[12] = {
    1.93861300091875771e-01, 4.78080369979300202e-01, -1.85163134573934129e-01, -3.15745193379613209e-02,
    1.40862568085704715e-01, -1.32543619759139197e-01, 2.74017194880180233e-02, 1.19121362382883136e-01,
    -2.26096713052116927e-01, 2.21406339543712638e-01, -1.10008955300923306e-01, 8.88054390278034469e-03};
__constant__ double c_exp64[12] = {
    1.00000000000000000e+00, 1.00000000000000000e+00, 5.00000000000001887e-01, 1.66666666666666796e-01,
    4.16666666664879531e-02, 8.33333333331958900e-03, 1.38888889523528631e-03, 1.98412698900764028e-04,
    2.48014854415613131e-05, 2.75572408872298695e-06, 2.76326547225277896e-07, 2.51100492048186583e-08};

// G and G' of both pairs at t = x - 3/2 (x < X64): four independent Horner chains.
__device__ __forceinline__ void g64_near(double t0, double t1, double &G0, double &Gp0, double &G1, double &Gp1)
{
  double g0 = c_g64[NG64 - 1], g1 = g0, p0 = c_gp64[NG64 - 1], p1 = p0;
#pragma unroll
  for (int k = NG64 - 2; k >= 0; k--) {
    g0 = fma(g0, t0, c_g64[k]);
    g1 = fma(g1, t1, c_g64[k]);
    p0 = fma(p0, t0, c_gp64[k]);
    p1 = fma(p1, t1, c_gp64[k]);
  }
  G0 = g0, Gp0 = p0, G1 = g1, Gp1 = p1;
}

// 1/sqrt(x) from the hardware estimate and one cubic step (x > 0 and finite).
__device__ __forceinline__ double rsqrt64(double x)
{
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// The far form's coefficients, read through a pointer the compiler cannot see through: it would
// otherwise keep all 24 doubles in scalar registers across the pair loop beside the 34 of the near
// polynomials, and spill both to vector lanes (one readlane an instruction).
using ConstF64 = const double __attribute__((address_space(4))) *;  // scalar loads
__device__ __forceinline__ ConstF64 here(const double *q)
{
  ConstF64 p = (ConstF64)q;
  asm volatile("" : "+s"(p));
  return p;
}

// a b + c with c in scalar registers (left to the compiler, a coefficient used once is copied to
// vector registers first: two moves a multiply-add).
__device__ __forceinline__ double fma_sc(double a, double b, double c)
{
  double d;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
  return d;
}

// An exponent of exp64_neg: what lies beyond 800 is 800 there.  NaN stays NaN, as it does in exp (fmin
// would make 800 of it, and a body with a NaN coordinate would add 0).
__device__ __forceinline__ double exp64_arg(double x) { return x > 800.0 ? 800.0 : x; }

// e^{-x} for 0 <= x <= 800 (0 from x = 745 on).  c: c_exp64, or here(c_exp64) where the call is rare.
template <class C> __device__ __forceinline__ double exp64_neg(double x, C c)
{
  const double k  = rint(x * -1.4426950408889634);
  const double r  = fma(k, -2.3190468138462996e-17, fma(k, -0.6931471805599453, -x))  /* ln 2 in two parts */;
  double       p  = c[NEXP64 - 1];
#pragma unroll
  for (int i = NEXP64 - 2; i >= 0; i--) p = fma_sc(p, r, c[i]);
  return __builtin_amdgcn_ldexp(p, (int)k);
}

// G, G' (and D2: G'') at x >= X64.
template <bool D2>
__device__ __forceinline__ void g64_far(double x, double &G, double &Gp, double &Gpp)
{
  const double w = rsqrt64(x), w2 = w * w;
  double       g = 1.0, ce = 0.0;
  if (x < FAR64) {
    // (the minimum is for the instruction schedule alone: without it the coefficients' scalar loads move
    // next to their first use, and the direct sum takes 2% longer)
    const double e = exp64_neg(fmin(x, 800.0), here(c_exp64)), t = fmax(w, FAR64_WMIN) - FAR64_WC;
    const ConstF64 c = here(c_far64);
    double         p = c[NFAR64 - 1];
#pragma unroll
    for (int k = NFAR64 - 2; k >= 0; k--) p = fma_sc(p, t, c[k]);
    g  = fma(-e, fma(TWO_SQRTPI, x * w, p), 1.0);
    ce = TWO_SQRTPI * e;
  }
  G  = g * w2 * w;
  Gp = w2 * fma(-1.5, G, ce);
  if (D2) Gpp = w2 * fma(-2.5, Gp, -ce);
}

// q = 1 / (2 sigma^2) of the FP64 factors.  The powers of q that scale G, G' and G'' (to q^{7/2}) stay in
// range with G itself (from x^{-3/2} down) for q <= Q64_MAX; a smaller core (sigma < 7e-36) acts as
// that one, with the same factors from R = 7e-35 on, where g = 1 either way.  A core without a kernel
// (sigma = 0 or NaN, so q infinite or NaN) is marked by a negative q: a coincident pair is still skipped,
// and any other takes a polynomial far outside its range, to infinity or NaN.
constexpr double Q64_MAX = 1e70;
__device__ __forceinline__ double core_q64(double sg)
{
  const double q = 0.5 / (sg * sg);
  return q < INFINITY ? fmin(q, Q64_MAX) : -Q64_MAX;
}
// |q|^{3/2}
__device__ __forceinline__ double pow32(double q) { return fabs(q) * sqrt(fabs(q)); }

// G and G' of two pairs at x = R^2 q.  A coincident pair (R^2 = 0) is skipped
// (multipoleKernels.hpp:242): only the f1 alpha terms survive a zero separation, so G = 0 is enough.
// The common path is taken where both x lie in (0, X64), one unsigned test of each high word (x
// below 2^-1022 counts as 0 there and is looked at again, and so is x <= -0, of a negative q).
__device__ __forceinline__ void g64_pair2(double r20, double r21, double q0, double q1, double &G0, double &Gp0,
                                          double &G1, double &Gp1)
{
  const double x0 = r20 * q0, x1 = r21 * q1;
  const int    h0 = __double2hiint(x0), h1 = __double2hiint(x1), far = (int)X64_HI;
  G0 = G1 = Gp0 = Gp1 = 0.0;
  if (min(h0, h1) < far) g64_near(x0 - 0.5 * X64, x1 - 0.5 * X64, G0, Gp0, G1, Gp1);
  if (max((unsigned)h0 - 1u, (unsigned)h1 - 1u) >= X64_HI - 1u) {
    double d2;
    if (h0 >= far) g64_far<false>(x0, G0, Gp0, d2);
    if (h1 >= far) g64_far<false>(x1, G1, Gp1, d2);
    if (r20 == 0.0) G0 = 0.0;
    if (r21 == 0.0) G1 = 0.0;
  }
}

// Targets per pass of a near-field workgroup of BLK lanes over a leaf of nt targets: lanes are
// (target, source split) with S = BLK / ntp splits, and the leaf takes ceil(nt / ntp) passes over
// its source list.  With BLK = 256 a pass costs about 1/S of the list per lane plus the staging
// (about 1/128), so ntp = ceil(nt / np) with np in 1..8 minimising np (1/S + 1/128); e.g. nt = 200
// takes 4 passes of 50 targets and 5 splits (98% of the lanes busy) instead of one pass with 56
// idle lanes.  With BLK = 64 a 64-source chunk is too short to pay for its staging again: one pass.
template <int BLK>
__device__ __forceinline__ int near_targets_per_pass(int nt)
{
  int best = max(1, min(nt, BLK));
  if (BLK <= 64) return best;
  float cost = 3.0e38f;
  for (int np = 1; np <= 8; np++) {  // np = 1 gives best, with cost 1/S + 1/128
    const int ntp = max(1, (nt + np - 1) / np);
    if (ntp > BLK) continue;
    const float c = np * (1.0f / (float)(BLK / ntp) + 1.0f / 128.0f);
    if (c < cost) cost = c, best = ntp;
  }
  return best;
}

// Source splits of a pass of ntp targets; 2 S entries must fit in half a staged chunk (BLK <= 64
// stages 2 BLK entries, BLK = 256 stages 256).
template <int BLK> __device__ __forceinline__ int near_splits(int ntp) { return min(BLK / ntp, BLK <= 64 ? 64 : 128); }

constexpr int SEG = 256;  // source leaves whose prefix sums sit in LDS at once

// Exclusive prefix sum of v[0..n) (n <= SEG) into pref[0..n]; one wavefront, 4 per lane.
__device__ __forceinline__ void lds_prefix(int *pref, const int *v, int n)
{
  const int lane = threadIdx.x;
  int       loc[4], tot = 0;
  for (int k = 0; k < 4; k++) {
    const int i = 4 * lane + k;
    loc[k]      = i < n ? v[i] : 0;
    tot += loc[k];
  }
  int incl = tot;
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(incl, o, 64);
    if (lane >= o) incl += u;
  }
  int run = incl - tot;
  for (int k = 0; k < 4; k++) {
    const int i = 4 * lane + k;
    if (i <= n) pref[i] = run;
    run += loc[k];
  }
  if (lane == 63 && 256 <= n) pref[256] = run;
}

// Body g of the list entries whose leaf sizes have the prefix sums pref[0..n] and first bodies lb:
// that of the last entry q with pref[q] <= g.
__device__ __forceinline__ int64_t list_body(const int *pref, const int *lb, int n, int g)
{
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (pref[mid] <= g) lo = mid;
    else hi = mid - 1;
  }
  return lb[lo] + (g - pref[lo]);
}

}  // namespace
}  // namespace uvlm
