// rules.hpp -- bounds and launch rules that are plain arithmetic on the host (no HIP).
#pragma once
#include <stdint.h>

namespace tg {

// Relative slack kappa of a screen distance s = (|a|^2 + |b|^2) - 2 a'.b':
// |s - d| <= kappa (|a|^2 + |b|^2), d the canonical FP32 distance; |a| |b| <= (|a|^2 + |b|^2) / 2.
//
// Products: nothing is assumed about the order of an MFMA step's additions, about intermediate
// rounding (to nearest or cut off) or about addends cut to the unit of the largest one: each
// addend costs at most 2^-23 of the absolute sum.  A step adds its products and the running
// sum, 33 addends for 32 elements of 16-bit rows, 5 for 4 elements of FP32 rows, so a' . b' is
// off by 33 D / 32 (5 D / 4) units of 2^-23 |a| |b|, and s by as many of |a|^2 + |b|^2.  (FP32
// chains on the vector unit add fewer.)  A kernel that sums chains of `chain` elements by FP32
// additions is off by 33 chain / 32 + D / chain.  The canonical fold costs D / 64 + 14 units of
// 2^-24 of d <= 2 (|a|^2 + |b|^2), the norms, s and the two ends of the interval a few more:
// below 128 units of 2^-23 for D <= 1024.  Rows whose |x|^2 is below 2^-96 are outside this
// (their products are not normal FP32 numbers).
//
// 16-bit rows: rho bounds |x' - x| / |x| over the rows (0 for exact copies), which puts the
// product off by at most (2 rho + rho^2) |a| |b|.
inline float screen_kappa16(double rho, uint32_t D, uint32_t chain) {
  const double q = (2.0 * rho + rho * rho) * (1.0 + rho) * (1.0 + rho);
  const double sum = D <= chain ? 33.0 / 32.0 * D : 33.0 / 32.0 * chain + (D + chain - 1) / chain;
  return float((q + (sum + 128.0) / 8388608.0) * (1.0 + 1e-5));
}
inline float screen_kappa32(uint32_t D) { return float((1.25 * D + 128.0) / 8388608.0); }

}  // namespace tg
