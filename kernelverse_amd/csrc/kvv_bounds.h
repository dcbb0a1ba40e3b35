// Bounds and rules shared by the device code and the host checks of the tests
// (plain C++: no HIP types, so g++ builds it too).
#pragma once

#include <math.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define KVV_HD __host__ __device__
#else
#define KVV_HD
#endif

namespace kvv {

// The keys of one select round's cell that the final read-off reads: the
// round's table gives the cell's start (t_lo) and the next cell's start (t_hi).
// Both are clamped to the round's own sample count (`chunk` samples per round,
// fewer in a group's last round), so lo + len never passes the round's span of
// the sample array, whatever the table words hold.
struct CellSpan {
  uint32_t lo, len;
};

KVV_HD inline CellSpan cell_span(uint32_t t_lo, uint32_t t_hi, int64_t count, int64_t round, int64_t chunk) {
  const int64_t left = count - round * chunk;
  const uint32_t rsz = left <= 0 ? 0u : (left < chunk ? (uint32_t)left : (uint32_t)chunk);
  uint32_t lo = t_lo < rsz ? t_lo : rsz;
  uint32_t len = t_hi - t_lo;  // wraps when the words are out of order: the clamp below bounds it
  len = len <= rsz - lo ? len : rsz - lo;
  return CellSpan{lo, len};
}

// floor(x / d) for every x < 2^31 (2 <= d < 2^31) as mulhi(x, mul) >> sh: with l
// = ceil(log2 d), mul = floor(2^(31 + l) / d) + 1 fits 32 bits, mul * d exceeds
// 2^(31 + l) by at most d <= 2^l, and x * 2^l < 2^(31 + l), so the quotient is exact.
KVV_HD inline void row_magic(uint32_t d, uint32_t& mul, uint32_t& sh) {
  uint32_t l = 1;
  while (l < 31 && (1u << l) < d) ++l;
  mul = (uint32_t)((1ull << (31 + l)) / d + 1);
  sh = l - 1;
}

// The one-compare form of the isclose test (abs_diff <= fl(atol + fl(rtol * |g|)),
// or g == r): abs_diff < fma(|g|, rtol_lo, atol_lo) holds for close pairs only,
// and for every finite pair of equal values.
//
// x_lo = fl(x * (1 - 2^-21)) <= x * (1 - 2^-22), so before its one rounding the
// bound is at most (X + A) * (1 - 2^-22), X = rtol * |g| and A = atol; the exact
// bound is at least (X + A) * (1 - 2^-24) - 2^-150.  For A >= 2^-127 the first is
// the smaller, and for A = 0 rounding's monotonicity orders them.  A bound of at
// least q = 2^-149, the least positive float, lets the equal pairs pass: where the
// floats are multiples of q (below 2^-125), fl(X_lo + q) = fl(X_lo) + q, and an
// abs_diff below it is at most fl(X_lo); above, q is less than the margin.
// Tolerances outside [2^-100, 2^100] (zero aside) and a zero tolerance (plain
// equality) leave q alone: only equal values pass.  An infinite abs_diff, and
// that of equal infinities (NaN), never do.
struct LeanTol {
  float rtol, atol;
};

KVV_HD inline LeanTol lean_tol(float rtol, float atol, bool zero_tol) {
  const float q = 0x1p-149f;
  const bool r_ok = rtol == 0.0f || (rtol >= 0x1p-100f && rtol <= 0x1p100f);
  const bool a_ok = atol == 0.0f || (atol >= 0x1p-100f && atol <= 0x1p100f);
  if (zero_tol || !r_ok || !a_ok) return LeanTol{0.0f, q};
  const float a = atol * (1.0f - 0x1p-21f);
  return LeanTol{rtol * (1.0f - 0x1p-21f), a > q ? a : q};
}

KVV_HD inline bool lean_close(float abs_diff, float g, float rtol_lo, float atol_lo) {
  return abs_diff < fmaf(fabsf(g), rtol_lo, atol_lo);
}

// Whether an item of `pairs` pairs, `slow` of them differing or not finite, is
// finished as a dense one, where at least 1 / kDenseShare of them are slow.  Of
// `lanes` of the slow pairs, `pass` pass the one-compare test, `miss` are finite
// and fail it, and the others are not finite.
//
// A dense item costs about as much as 7 (16-bit) or 3 (fp32) queue steps of 64
// slow pairs, i.e. a quarter of the item's, and saves the steps of the pairs that
// pass; those that fail go to the queue all the same, except that fp32's
// mismatches are mostly counted in place (half a step's share).  Next to pairs
// that are not finite, whose steps take twice as long, a pair that passes saves
// twice as much; in a capture segment the queue's steps capture too, which those
// of a dense item's rest do not.
//
// With every item of a quarter slow pairs dense, as it was first, verdicts that
// fail took longer than through the queue.  32 Mi pairs, us by the queue, by every
// such item dense, and by this rule: a quarter of the pairs beyond the tolerance
// (the others identical) fp32 112, 141, 113 and bf16 92, 142, 94; a half, bf16 128,
// 170, 130; zero tolerance and a half of the pairs different, fp32 136, 174, 136 and
// bf16 98, 168, 100; half of the pairs -inf, the others identical, bf16 179, 198, 181.
constexpr uint32_t kDenseShare = 4;
KVV_HD inline bool dense_pays(bool fp32, bool capture, uint32_t slow, uint32_t pairs, uint32_t lanes, uint32_t pass,
                              uint32_t miss) {
  const uint32_t other = lanes - pass - miss;
  const uint32_t gain = 2 * pass * (other * 8 >= lanes ? 2 : 1) + (fp32 ? miss : 0) + (capture ? other : 0);
  const uint32_t need = !fp32 && miss * 16 >= lanes ? 5 : 4;  // (the look for the failing pairs costs as much as two steps)
  return slow * gain * (2 * kDenseShare) >= need * lanes * pairs;
}

// fp32 items of at least three quarters slow pairs need no look at them: dense costs
// them less than the queue whatever they are (all beyond the tolerance: 32 Mi pairs
// 144 us, 201 with every mismatch in the queue).  The look at one pair per lane takes
// 0.3 us of the verdict of a few thousand elements.
KVV_HD inline bool dense_surely_pays(bool fp32, uint32_t slow, uint32_t pairs) { return fp32 && slow * 4 >= 3 * pairs; }

// Whether the item after a dense one that left `rest` of its `pairs` pairs to
// the queue is taken as dense without being classified.  (fp32: always, the rest
// costs it no more than the queue would.)
KVV_HD inline bool dense_goes_on(bool fp32, uint32_t rest, uint32_t pairs) { return fp32 || rest * 4 < 3 * pairs; }

}  // namespace kvv
