// Host check of csrc/rate_groups.h: prints the first fault and returns 1, or
// prints the number of grids checked.
#include "rate_groups.h"

#include <cstdio>
#include <initializer_list>

using namespace zdt;

// the parts of n groups take every group once, and none is empty
static bool tiles(int n, unsigned np) {
  if (np < 1 || group_first(n, 0, np) != 0 || group_first(n, np, np) != n) return false;
  for (unsigned y = 0; y < np; ++y)
    if (group_first(n, y, np) >= group_first(n, y + 1, np)) return false;
  return true;
}

int main() {
  const int shapes[][2] = {{64, 512},  {64, 1024},  {128, 512}, {128, 1024},
                           {256, 512}, {256, 1024}, {512, 512}, {512, 1024}};  // N1, N2
  long n = 0;
  for (const auto& s : shapes)
    for (int paired = 0; paired < 2; ++paired)
      for (int Nr = 1; Nr <= 1200; ++Nr)
        for (int64_t ncu : {64, 256, 304}) {
          int units = 0;  // pairs (j, Nr-1-j), j <= Nr-1-j, or rates
          for (int j = 0; j < Nr; ++j) units += !paired || j <= Nr - 1 - j;
          const int per = k2_rows(s[0]) / (paired ? 4 : 2);
          const int ng = k2_groups(Nr, k2_rows(s[0]), paired != 0);
          const unsigned np = k2_parts(s[0], s[1], ng, ncu);
          if (ng * per < units || (ng - 1) * per >= units || !tiles(ng, np)) {
            std::printf("k2 N1=%d N2=%d paired=%d Nr=%d: %d groups for %d units, %u parts\n", s[0], s[1], paired, Nr,
                        ng, units, np);
            return 1;
          }
          ++n;
        }
  // the other kernels' rules (least groups a part, wavefronts a CU) up to 2^24 rates
  const int rules[][3] = {{256, 12, 8}, {256, 12, 20}, {256, 8, 24}, {256, 16, 8}, {64, 24, 2}, {1024, 16, 1}};
  for (const auto& r : rules)
    for (int nblk : {1, 2, 3, 17, 256, 1024})
      for (int ng : {1, 2, 7, 8, 63, 65535, 65536, 5592405, 5592406, 8388607, 8388608, 16777216})
        for (int64_t ncu : {64, 256, 304}) {
          const unsigned np = group_parts(ng, nblk, r[0], r[1], r[2], ncu);
          if (np > 65535 || !tiles(ng, np)) {
            std::printf("%d groups, %d blocks of %d: %u parts\n", ng, nblk, r[0], np);
            return 1;
          }
          ++n;
        }
  std::printf("%ld grids\n", n);
  return 0;
}
