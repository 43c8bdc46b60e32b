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
// below 128 units of 2^-23 for D <= 1024.  Products below the smallest normal FP32 number may
// count as 0, 2^-115 together, which is in the slack of rows with |x|^2 >= 2^-96; smaller rows
// have no norm (k_screen_prep), and every comparison with their s leaves the pair undecided.
//
// 16-bit rows: rho bounds |x' - x| / |x| over the rows (0 for exact copies), which puts the
// product off by at most (2 rho + rho^2) |a| |b|.
inline float screen_kappa16(double rho, uint32_t D, uint32_t chain) {
  const double q = (2.0 * rho + rho * rho) * (1.0 + rho) * (1.0 + rho);
  const double sum = D <= chain ? 33.0 / 32.0 * D : 33.0 / 32.0 * chain + (D + chain - 1) / chain;
  return float((q + (sum + 128.0) / 8388608.0) * (1.0 + 1e-5));
}
inline float screen_kappa32(uint32_t D) { return float((1.25 * D + 128.0) / 8388608.0); }

// Slots (log2) of a search workgroup's visited hash in LDS: two thirds filled at the usual
// L * FD / 2 + L visited ids, 2^10 to 2^13, but no more than leaves room for `per_cu` workgroups
// in a CU's 160 KB (allocated in units of 1,280 bytes; SEARCH_LDS besides the hash).  A search
// that fills its hash goes on in a bitmap in device memory, which costs less than waves that do
// not run.  10,000 queries, 12 or (all rows above 256 elements, u8 rows above 128) 8 workgroups
// per CU, at the largest size / at this one: 200k x 96 FP32 rows, FD 32, L 256 10.9 / 5.5 ms, FD
// 48, L 128 5.7 / 3.2; 300k x 128 u8 rows, FD 32, L 256 8.2 / 4.3; 100k x 256 u8 rows, FD 48, L
// 128 4.3 / 2.9; 50k x 960, FD 48, L 128 8.9 / 6.9.  1,000 queries (4 per CU), 300k x 128, FD
// 48, L 128: 0.64 ms at 2^13, 0.80 at 2^11.
constexpr uint32_t SEARCH_LDS = 256 * 8 + 256 * 4 + 64 * 4;
inline uint32_t search_hash_bits(uint32_t L, uint32_t FD, uint32_t per_cu) {
  const uint32_t usual = L * FD / 2 + L + 128;
  uint32_t bits = 10;
  while (bits < 13 && (2u << bits) < 3 * usual) ++bits;
  auto lds = [](uint32_t b) { return ((4u << b) + SEARCH_LDS + 1279) / 1280 * 1280; };
  while (bits > 10 && per_cu * lds(bits) > 160 * 1024) --bits;
  return bits;
}

}  // namespace tg
