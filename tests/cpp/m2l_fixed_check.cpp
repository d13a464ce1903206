// Host check of the M2L plans that k_m2l_fixed is compiled for (uvlm_amd/csrc/m2l_plan.hpp): each
// table is the plan of its order for the default budget, no other budget's plan of another
// structure is taken for it, and where a home slot reads M[n, m] from its lanes' registers the
// lanes 0..n are active in it.  Exit status 0 when all hold.
#include "../../uvlm_amd/csrc/m2l_plan.hpp"

#include <cstdio>
using namespace uvlm;
int main()
{
  int bad = 0, fixed = 0;
  for (int P = 1; P <= 16; P++) {
    const M2LFixed f = m2l_fixed(P);
    if (!f.S) continue;
    fixed++;
    M2LPlan pl;
    if (!make_m2l_plan(P, f.W == 2 ? 5 : 0, pl, 16, f.W) || !m2l_plan_fixed(pl)) { printf("P=%d: not the default plan\n", P); bad++; }
    for (int W : {1, 2})
      for (int b : {0, 4, 5, 6, 8, 12, 16}) {
        M2LPlan o;
        if (!make_m2l_plan(P, b, o, 16, W)) continue;
        const bool same = o.S == f.S && o.W == f.W && o.lev == pl.lev;
        if (m2l_plan_fixed(o) != same || (same && o.slots != pl.slots)) { printf("P=%d W=%d b=%d taken\n", P, W, b); bad++; }
      }
    for (int w = 0; w < f.W; w++)
      for (int n = 0; n < P; n++) {
        const int lv = f.lev[w * P + n], hr = (lv >> 8) & 255, A = plan_tri(P - n);
        if (hr > f.home(w)) bad++;
        for (int s = 0; s < hr; s++) {
          int active = 0;  // lanes 0 .. active - 1
          while (active < 16 && 16 * s + active < A) active++;
          if (m2l_row(A, s, n) && active <= n) { printf("P=%d n=%d s=%d: %d lanes\n", P, n, s, active); bad++; }
          if (active == 0) { printf("P=%d n=%d s=%d: empty round\n", P, n, s); bad++; }
        }
      }
  }
  printf("%d orders, %s\n", fixed, bad ? "FAILED" : "all match");
  return bad != 0 || fixed == 0;
}
