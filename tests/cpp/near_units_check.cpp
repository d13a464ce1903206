// Host check of the near-field unit arithmetic (uvlm_amd/csrc/near_units.hpp): the units, the
// leaves cut into several and their partial sums never pass what is reserved or allowed for them, and a
// leaf's units cover its list.
// Work totals just above and just below each multiple of UNITS_AIM, spread over few leaves, over many,
// and over a few among thousands that have none.  Exit status 0 when all hold.
#include "../../uvlm_amd/csrc/near_units.hpp"

#include <cstdio>
#include <vector>
using namespace uvlm;
int main()
{
  int  bad = 0;
  long sets = 0;
  const auto check = [&](const std::vector<uint32_t> &work, int len, const char *what, int nt = 1,
                         uint64_t allowed = UNITS_ROWS_MAX) {
    uint64_t total = 0;
    for (uint32_t w : work) total += w;
    const uint64_t lim   = units_limit(total, nt * total, allowed);
    const int64_t  nleaf = (int64_t)work.size();
    int64_t        units = 0, multi = 0, rows = 0;
    for (uint32_t w : work) {
      const int n = units_of_leaf(w, len, lim);
      units += n;
      multi += n > 1;
      rows += n > 1 ? (int64_t)n * nt : 0;
      bool covered = units_first(len, 0, n) == 0 && units_first(len, n, n) == len;
      for (int j = 0; j < n && nleaf < 100; j++) covered = covered && units_first(len, j, n) <= units_first(len, j + 1, n);
      if (n < 1 || !covered) { printf("%s: %d units of a list of %d\n", what, n, len); bad++; }
    }
    if (units > units_bound(nleaf) || multi > units_multi_bound(nleaf) || rows > (int64_t)allowed) {
      printf("%s: %ld leaves, %llu steps: %ld units, %ld cut, %ld rows\n", what, (long)nleaf, (unsigned long long)total, (long)units,
             (long)multi, (long)rows);
      bad++;
    }
    sets++;
  };
  for (uint64_t k : {1, 2, 63, 64, 65, 66, 100, 127, 1000, 65535})
    for (int64_t add : {-1, 0, 1, 14746, 16382, 16383}) {
      const uint64_t total = k * UNITS_AIM + add;
      for (int heavy : {1, 2, 60, 199, 700})
        for (int rest : {0, 1, 4040, 20000}) {
          if (total / heavy >= (uint64_t(1) << 32)) continue;
          std::vector<uint32_t> work(heavy + rest, 0);
          for (int i = 0; i < heavy; i++) work[i] = (uint32_t)(total / heavy + (i < (int)(total % heavy)));
          check(work, 1 << 20, "few leaves with work");
          for (int nt : {192, 1000, 40000})
            for (uint64_t rows : {UNITS_ROWS_MAX, uint64_t(1000001), uint64_t(3), uint64_t(0)})
              check(work, 1 << 20, "few leaves of many targets", nt, rows);
          check(work, 3, "short lists");
        }
      for (int nleaf : {16384, 16500, 40000}) {  // every leaf a little over the limit's share
        std::vector<uint32_t> work(nleaf);
        for (int i = 0; i < nleaf; i++) work[i] = (uint32_t)(total / nleaf + (i < (int)(total % nleaf)));
        check(work, 1 << 20, "all leaves alike");
        check(work, 1 << 20, "all leaves alike, of many targets", 900);
      }
    }
  check({}, 0, "no leaves");
  check({0}, 0, "an empty list");
  check({0xffffffffu, 0xffffffffu, 1}, 1 << 30, "the largest work");
  printf("%ld sets, %s\n", sets, bad ? "FAILED" : "all within their buffers");
  return bad != 0 || sets == 0;
}
