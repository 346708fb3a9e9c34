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

}  // namespace bfe
