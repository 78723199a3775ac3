// First pass of the merged selection of window-key scores (listbuild.hip): bins of equal width over the bulk of a row.
//
// The scores are sums of signed products, so the top bits of their keys (sign, exponent, two bits of mantissa) fill a few
// dozen bins and the bin of the threshold holds several hundred keys of 10521: two more passes.  Bins of equal width hold a
// few dozen keys at most, but between the smallest and the largest score they do so only while no score lies far from the
// others: one that does leaves the others in a handful of bins, whose counts then serialise, and the pass is lost.  So the
// bins span twice the range that every group of neighbouring threads reaches: the smallest of the largest keys
// of a group's threads, over the groups the largest.  Keys beyond it count in the end bins.  A far score changes it only
// where it comes with one in every thread of a group; of normal scores it is 1.5 .. 2 standard deviations each way.  Scores
// spread over many orders of magnitude have no such range: it differs by as much between waves, and the digits are as good
// as bins can be there.  32 rows of 10521 scores, 1792 kept; digits only / bins from the smallest to the largest / these, us:
// normal 16.0 / 12.1 / 11.9, one score 100 times the others 16.0 / 24.1 / 12.0, two at +-1e30 16.0 / 28.3 / 11.9, a hundredth
// of them far 16.1 / 24.1 / 11.9, a Cauchy distribution 20.0 / 31.1 / 12.3, exp(12 |x|) 13.6 / 26.0 / 14.8.
// Arithmetic shared by the device code and by a host-side test.
#pragma once
#include <stdint.h>

#ifndef LVAR_HD
#if defined(__HIPCC__)
#define LVAR_HD __host__ __device__ __forceinline__
#else
#define LVAR_HD inline
#endif
#endif

namespace lvar {

constexpr int SCORE_BINS = 2048;
constexpr uint32_t KEY_NEG_INF = 0x007fffffu, KEY_POS_INF = 0xff800000u;   // real_key of -inf and +inf

// Threads of a group, a power of two: the fewer keys a thread has, the lower the smallest of the group's largest keys.
constexpr int score_group(int keys_per_thread) { return keys_per_thread >= 8 ? 8 : keys_per_thread >= 4 ? 4 : 2; }

LVAR_HD float score_of_key(uint32_t key) {
  union { uint32_t u; float f; } x;
  x.u = key ^ ((key >> 31) ? 0x80000000u : 0xffffffffu);
  return x.f;
}

struct ScoreBins { float x0, xs; };

// Width of one wave's bulk [lo, hi], or 0 where it has none.
LVAR_HD float score_width(uint32_t lo, uint32_t hi) {
  return KEY_NEG_INF < lo && lo < hi && hi < KEY_POS_INF ? score_of_key(hi) - score_of_key(lo) : 0.f;
}

// Bins for a bulk of [lo, hi] whose narrowest full wave has a bulk of width `narrow`, or false where it is empty, not finite,
// spread over orders of magnitude, or so narrow that 1 / width is not finite.
LVAR_HD bool score_bins(uint32_t lo, uint32_t hi, float narrow, ScoreBins& b) {
  const float width = score_width(lo, hi);
  union { float f; uint32_t u; } range;
  range.f = 2.f * width;
  if (range.u <= 0x08000000u || range.u >= 0x7f800000u) return false;   // 2^-111; infinite
  if (!(width <= 24.f * narrow)) return false;   // (of normal scores up to 6 times, with a mean that rises by 20 deviations 12, of exp(12 |x|) 27 and more)
  b.x0 = 0.5f * score_of_key(lo) + 0.5f * score_of_key(hi) - 0.5f * range.f;
  b.xs = (float)(SCORE_BINS - 1) / range.f;
  return true;
}

// Monotonic in the key (subtraction, product and truncation are): a bin is a run of keys.  A NaN stands where its key does,
// beyond the infinity of its sign.
LVAR_HD int score_bin(const ScoreBins& b, uint32_t key) {
  const uint32_t k = key < KEY_NEG_INF ? KEY_NEG_INF : key > KEY_POS_INF ? KEY_POS_INF : key;
  const float at = (score_of_key(k) - b.x0) * b.xs, last = (float)(SCORE_BINS - 1);
#if defined(__HIP_DEVICE_COMPILE__)
  return (int)__builtin_amdgcn_fmed3f(at, 0.f, last);
#else
  return (int)(at < 0.f ? 0.f : at > last ? last : at);
#endif
}

}  // namespace lvar
