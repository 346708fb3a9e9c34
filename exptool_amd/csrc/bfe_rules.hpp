// Rules that choose a kernel or a launch shape from sizes alone (host code, no
// HIP): plain functions, so that they can be walked over whole ranges on the
// CPU.  Every form a rule chooses between gives the same bits.
#pragma once

#include <cstdint>

namespace bfe {

// Builds of field_eval_kernel: 144 registers (three waves a SIMD) or 128 with
// 20 B spilled (four).  The second pays only where a fourth wave has work, from
// about eight blocks of 256 a CU.  Three / four, in cell order: 262 144 points
// 63.5 / 65.8 us at lmax = mmax = 6 and 90.2 / 95.0 at 12, 500 000 90.0 / 91.6 and
// 128.7 / 130.5, 800 000 115.6 / 113.9 and 173.7 / 168.3, 2M 218 / 214 and 342 /
// 320; in input order 65 536 points 22.6 / 24.0 and 47.9 / 56.6.
constexpr int64_t kEvalFourWaves = 524288;
inline bool eval_four_waves(int64_t n) { return n >= kEvalFourWaves; }

// Terms of one field evaluation: SL (l, m) pairs and EOF orders.
inline int field_terms(int lmax, int mmax) { return (lmax + 1) * (lmax + 2) / 2 + mmax; }
// Bases whose split kernels have their orders at compile time.
inline bool split_fixed(int lmax, int mmax) { return lmax == 6 && mmax == 6; }

// Orbits up to which the split integrators run (64 a block of eight waves, one
// block a CU: 16 384 orbits are one round of the 256 CUs, 32 768 two).  A round
// costs a fixed part whatever the basis; the one-lane kernels cost their terms
// (RK4 more of them a term) and nothing more up to 65 536 orbits.  So the second and
// third rounds pay from some number of terms on, where the orders are found at run
// time.  One lane / split in us at 16 384 | 32 768 | 36 864 orbits, (lmax, mmax):
//   leapfrog, 100 steps  (2, 2)  552 / 436 | 578 / 779     (4, 4) 833 / 514 | 814 / 909
//     (4, 6) 945 / 513 | 909 / 905     (6, 4) 1195 / 597 | 1182 / 1054 | 1167 / 1485
//     (10, 6) 1927 / 854 | 1926 / 1546 | 1903 / 2260     (6, 6) at its own instance
//     1294 / 480 | 1279 / 804 | 1274 / 1112
//   RK4, 25 steps  (3, 3) 892 / 525 | 876 / 956     (4, 2) 869 / 449 | 860 / 820
//     (5, 5) 1260 / 539 | 1233 / 986 | 1229 / 1391     (6, 0) 1305 / 467 | 1254 / 833 |
//     1254 / 1164     (10, 6) 2651 / 851 | 2586 / 1544 | 2603 / 2276
// At any other value than its default the knob is the limit for every basis.
constexpr int64_t kSplitMax = 36864;
inline int64_t split_orbits_max(int64_t knob, int lmax, int mmax, bool rk4) {
  if (knob != kSplitMax || split_fixed(lmax, mmax)) return knob;
  const int terms = field_terms(lmax, mmax);
  if (rk4 && terms >= 28) return kSplitMax;
  return terms >= (rk4 ? 15 : 21) ? 32768 : 16384;
}

}  // namespace bfe
