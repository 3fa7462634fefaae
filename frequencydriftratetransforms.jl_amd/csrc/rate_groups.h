// How the column-pair and chirp-Z kernels split their groups of rates (or time
// steps) over blockIdx.y where the columns or bins alone leave the chip idle.
// The host sizes the grid from the same group counts that the kernels walk:
// every part has at least one group, so no kernel needs a path for an empty one.
// Plain constexpr C++ for both sides.
#pragma once

#include <cstdint>

namespace zdt {

// groups of `per` in n
constexpr int groups_of(int n, int per) { return (n + per - 1) / per; }

// mirrored pairs of rates (j, Nr-1-j), the middle rate of an odd Nr a pair of its own
constexpr int rate_pairs(int Nr) { return (Nr + 1) / 2; }

// k2's rows per group: as many as keep one butterfly per lane in the
// wavefront-level passes (8 rows for 512 = 8*8*8 over 8 wavefronts, ...)
constexpr int k2_rows(int n1) { return n1 == 256 ? 16 : 8; }

// k2_czt's groups for `rows` rows in LDS: two rows a rate, four a pair of rates
constexpr int k2_groups(int Nr, int rows, bool paired) {
  return paired ? groups_of(rate_pairs(Nr), rows / 4) : groups_of(Nr, rows / 2);
}

// First of the n groups that part y of np takes (0 <= y <= np; n np < 2^32, which
// group_parts sees to).
constexpr int group_first(int n, unsigned y, unsigned np) {
  return static_cast<int>(static_cast<unsigned>(n) * y / np);
}

// Parts (blockIdx.y) for ng groups: as many as bring nblk blocks of `threads` up
// to `waves` wavefronts a CU, with at least `least` groups each.
constexpr unsigned group_parts(int ng, int nblk, int threads, int waves, int least, int64_t ncu) {
  int64_t s = waves * ncu / (static_cast<int64_t>(nblk) * (threads / 64));
  if (s > ng / least) s = ng / least;
  if (s > 0xFFFFFFFFll / ng) s = 0xFFFFFFFFll / ng;  // 5.6 million groups and more
  return static_cast<unsigned>(s < 1 ? 1 : s);
}

// k2_czt's parts.  Each part repeats the input phase, which costs nothing while
// the CUs have room (one wavefront per SIMD issues no slower beside others), so
// parts go down to one group: 2^16 channels 17 rates 21.3 -> 16.1 us against three
// groups at least, 9 17.3 -> 15.5, 33 19.9 -> 18.9, 2^18 x 65 42.2 -> 40.0; 2^17 x 33
// 22.9 -> 23.9.  The waves a CU holds are bounded by VGPRs (N1 <= 128) or LDS (256:
// 8, 512: 16).  At 129 rates, one part -> this rule: 2^16 69.8 -> 29.6 us, 2^17
// 72.6 -> 36.6, 2^18 93.0 -> 61.7; a second part only costs at 2^19 (110.8 ->
// 128.3) and 2^20 (181 -> 205), whose blocks fill the chip.
constexpr unsigned k2_parts(int N1, int N2, int groups, int64_t ncu) {
  return group_parts(groups, N2 / 2, N1 < 512 ? N1 : 512, N1 >= 512 ? 16 : (N1 == 256 ? 8 : 12), 1, ncu);
}

}  // namespace zdt
