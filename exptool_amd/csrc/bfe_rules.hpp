// Rules that choose a kernel or a launch shape from sizes alone (host code, no
// HIP): plain functions, so that they can be walked over whole ranges on the
// CPU.  Every form a rule chooses between gives the same bits.
#pragma once

#include <cstdint>

namespace bfe {

// Builds of field_eval_kernel: 144 registers (three waves a SIMD) or 128 with
// 20 B spilled (four).  The second pays only where a fourth wave has work, from
// about nine blocks of 256 a CU on.  Kernel us, three / four, in cell order at
// (lmax, mmax): 262 144 points (4, 4) 25.6 / 26.8, (6, 6) 32.6 / 34.9, (12, 12) 60.4 /
// 64.6; 524 288 38.6 / 39.6, 49.5 / 50.7, 88.2 / 90.8; 600 000 43.8 / 43.5, 55.8 /
// 56.5, 102.5 / 102.6; 800 000 53.4 / 51.5, 67.3 / 66.6, 125.8 / 121.8; 2M 108 / 102,
// 139 / 131, 260 / 244.  ((10, 6) and (2, 2) cross at 400 000: 58.3 / 56.6 there.)
// With cos(l phi) factors from six blocks a CU on: (10, 6) 300 000 61.6 / 63.5,
// 400 000 78.4 / 76.3, 600 000 102 / 98; (12, 12) 84.2 / 90.4, 106.7 / 106.0, 137 / 134.
constexpr int64_t kEvalFourWaves = 589824, kEvalFourWavesCosL = 393216;
inline bool eval_four_waves(int64_t n, bool cos_l) {
  return n >= (cos_l ? kEvalFourWavesCosL : kEvalFourWaves);
}

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

// The form of a field evaluation of n points: one lane a point in input order,
// split blocks (64 points a block of eight waves) or one lane a point in cell order
// (sorted first).
//
// One lane in input order is flat up to 65 536 points (a block of 256 a CU), then
// doubles.  The sort costs about 25 us, so it pays from the second round on where a
// point has many terms, from the third otherwise.  Split blocks cost with every
// round of theirs and win while one lane's latency is longer.  us in input order /
// split / cell order at (lmax, mmax) and points:
//   (2, 2)    16 384  7.7 / 10.1 / 29    65 536  9.0 / 32 / 31    131 072  14 / 57 / 36
//   (4, 4)    8 192 10.2 / 9.8 / 32    16 384 10.4 / 11.4 / 32    65 536 13 / 36 / 33
//             131 072  25 / 66 / 39
//   (4, 8)    16 384 14.2 / 13.7 / 34    24 576 17 / 23 / 34    131 072 42 / 76 / 46
//   (6, 6)    49 152  22 / 20.5 / 37    65 536  22.6 / 26.6 / 37    98 304 42 / 38 / 42
//             131 072  44 / 49 / 43
//   (8, 8)    32 768  33 / 29 / 40    65 536  33 / 52 / 41    80 000  60 / 63 / 48
//   (10, 6)   32 768  33 / 31 / 41    65 536  33 / 54 / 41    100 000  63 / 77 / 49
//   (12, 12)  32 768  48 / 40 / 52    65 536  48 / 72 / 58    100 000  102 / 104 / 69
//   without split blocks (cos(l phi)): (4, 4) 100 000 23 / - / 39, (6, 6) 42 / - / 45,
//   (10, 6) 62 / - / 58, (12, 12) 106 / - / 92
// (6, 6) is the split kernels' instance with its orders at compile time.
// At any other value than its default split_knob takes split blocks for every
// unordered call up to it.
enum EvalForm { kEvalInput = 0, kEvalSplit = 1, kEvalOrdered = 2 };
constexpr int64_t kSplitEvalMax = 131072;
constexpr int64_t kEvalRound = 65536;
inline EvalForm eval_form(int64_t n, int lmax, int mmax, bool split_ok, int64_t order_min,
                          int64_t split_knob) {
  const int terms = field_terms(lmax, mmax);
  const bool explicit_max = split_knob != kSplitEvalMax;
  if (!explicit_max && terms >= 45 ? n > order_min : n / 2 >= order_min) return kEvalOrdered;
  int64_t most = split_knob;
  if (!explicit_max) {
    if (split_fixed(lmax, mmax)) most = n <= kEvalRound ? 49152 : 98304;
    else most = terms >= 45 ? 32768 : terms >= 20 ? 16384 : 0;
  }
  return split_ok && n <= most ? kEvalSplit : kEvalInput;
}
// Whether the n points of two inputs are evaluated by split blocks or else ordered
// together (they have no one-lane form in input order): split / cell order at
// 49 152 | 57 344 points (0, 0) 20 / 28 | 25 / 28, (4, 4) 28 / 33 | 35 / 33, (6, 4) 31 /
// 36 | 39 / 36, (10, 6) 43 / 43 | 53 / 44, (12, 12) 57 / 63 | 71 / 62; (6, 6) at 114 688
// 44 / 46.
inline bool eval_split_two(int64_t n, int lmax, int mmax, bool split_ok, int64_t order_min,
                           int64_t split_knob) {
  if (!split_ok || n / 2 >= order_min) return false;
  if (split_knob != kSplitEvalMax) return n <= split_knob;
  return n <= (split_fixed(lmax, mmax) ? 114688 : 49152);
}

// Whether an input-order halo sum that has the GPU to itself takes the build of three
// blocks a CU: from more than two blocks a CU on, where three fit in the LDS.  us with
// two / three at (lmax, mmax): (6, 6) 30 000 particles (469 blocks) 25.4 / 26.3, 60 000
// 45.4 / 43.7; (8, 8) 60 000 45.6 / 43.7, 300 000 178.5 / 151.2, 1M 482 / 402; (10, 6),
// 54 KiB a block, 1M 521 / 532.
inline bool sl_three_blocks(int64_t blocks, uint64_t lds) { return blocks > 2 * 256 && 3 * lds <= 160 * 1024; }

// Nodes a group of four lanes folds in the whole-table SL fold: one until the lanes
// of two a group fill 128 blocks, then two, which share rows.  Whole calls, one / two,
// us at lmax, numr (nmax 20): 0, 2000 7.8 / 8.5; 2, 2000 10.3 / 11.0; 4, 1000 (30 000
// lanes) 13.2 / 13.8; 3, 2000 (40 000) 12.9 / 12.4; 6, 2000 22.1 / 20.4; 8, 4000 41.0 /
// 36.9.
inline int sl_fold_rows(int numr, int lmax) {
  return (int64_t)numr * (lmax + 1) * (lmax + 2) >= 32768 ? 2 : 1;
}

// Launch of the conservative surrogate's inference: the first `waves` of a block's
// eight take `per` 16-point tiles each at a time; at most one block a CU (its LDS
// holds the weights, loaded once by all eight: 1M points 523 us under a profiler,
// 537 with 2 048 blocks).  Up to 16 384 points four waves a block give every tile a
// SIMD to itself (14.8 us; eight on half the CUs 19.5); from there eight, and as many
// tiles a wave at a time as the waves of the whole device leave it, at most four
// (one point load and one base model a lane then serve four tiles), in rounds of
// nearly equal length.  32 769 points: two tiles a wave 30.8 us, four on a quarter of
// the CUs 54; 65 537: three 42.6, four 55.
struct GradLaunch {
  int waves, per, blocks;
};
inline GradLaunch mlp_grad_launch(int64_t n) {
  const int64_t tiles = (n + 15) / 16;
  const int waves = tiles <= 256 * 4 ? 4 : 8;
  const int64_t steps = (tiles + 256 * 8 - 1) / (256 * 8), rounds = (steps + 3) / 4;
  const int per = (int)((steps + rounds - 1) / rounds);
  const int64_t blocks = (tiles + (int64_t)per * waves - 1) / ((int64_t)per * waves);
  return GradLaunch{waves, per, (int)(blocks < 256 ? blocks : 256)};
}

// Blocks of the surrogate integrator: 16 orbits a wave with conservative forces (32
// without), four waves a block while that leaves one block a CU, then eight, whose
// waves cover each other but spill.  A step of 64 orbits 12.1 us with four (13.9 with
// eight), of 1 000 to 16 384 orbits 12.5 (30 with two tiles a block), of 32 768 17 (31).
// 2 048 blocks at most, eight a CU (256 at 1M orbits the same within 1 %).
struct LeapLaunch {
  int waves, blocks;
};
inline LeapLaunch mlp_leap_launch(int64_t n, bool conservative) {
  const int waves = conservative && n <= 256 * 4 * 16 ? 4 : 8;
  const int64_t pts = waves * (conservative ? 16 : 32), blocks = (n + pts - 1) / pts;
  return LeapLaunch{waves, (int)(blocks < 2048 ? blocks : 2048)};
}

}  // namespace bfe
