// Which form of workgroup a plain attention launch takes, by its sizes alone: host arithmetic, shared by the launch code and a
// host-side test.  All forms of a launch give the same bits.
#pragma once
#include <stdint.h>

namespace lvar {

inline int64_t workgroups(int64_t slices, int Lq, int rows) { return slices * ((Lq + rows - 1) / rows); }

// Pairs of waves with four fetch waves, where 64-row workgroups of them have a compute unit each.  128-row
// workgroups with four fetch waves / 64-row ones of pairs, B2 H16 d128: 36 x 85 5.82 / 5.53 us, 64 x 149 6.73 / 6.10, 144 x 265
// 8.78 / 7.42, 256 x 521 11.9 / 9.87, 400 x 921 16.8 / 13.8, 256 x 1497 23.7 / 18.7; B1 H4 4096 x 10521 134 / 120; d64 B1 H16
// 256 x 680 10.7 / 9.0; lists alike (B1 H8 576 x 1497 at 30 % 14.2 / 11.3, sink + window B1 H4 3025 x 9450 31.6 / 25.2); a single key
// tile alike; head_dim 256, where the waves of 128-row workgroups fill their SIMDs and nothing only fetches: 16 x 21 6.9 / 5.0,
// 144 x 265 15.1 / 10.2, 400 x 921 30.5 / 21.5, 512 x 1000 32.1 / 24.1, B1 H4 3000 x 9000 213 / 137.  Not beyond: pairs that share their SIMDs take twice
// as long (96-row workgroups of three pairs, 576 x 1497 24.3 / 25.8, 6000 x 10521 136 / 165; 128-row ones 24.4 / 29.6).  Two streams
// with such a launch each, B1 d128: 2 x 8 heads 576 x 1497 23.7 / 23.1, 2 x 16 heads 25.3 / 24.7, 2 x 8 heads 1024 x 2521 72.7 / 55.5,
// but 2 x 16 heads, which fill the chip together as 128-row workgroups, 51.2 / 64.9 (one stream 40.5 / 33.0).
// Lists of 64-row query blocks, token lists in groups that are no multiple of 192 rows and all token lists at head_dim 256 do not
// come here: they run as 2- and 3-wave workgroups that fetch for themselves, and have not been timed in pairs.
inline bool pairs_of_waves(int64_t slices, int Lq, int cus) { return workgroups(slices, Lq, 64) <= cus; }

// 256 query rows per workgroup (eight waves on one pair of K/V buffers, one workgroup per compute
// unit): half the L2->LDS fills per flop, 4 % faster than two 128-row workgroups side by side (B2 H16 d128: 4096 x 10521
// 635 -> 608 us, 1600 x 4121 117 -> 113 us) unless the coarser tiles leave more of the last round idle.  In units of a
// lone 128-row tile: a pair of 128-row workgroups takes 1.6 of it, a 256-row one 1.6 * 0.95; at head_dim 64 three small
// workgroups share a compute unit and only launches of a single round gain.  Lists of 256-row query blocks run the same way.
inline bool wide_tiles(int64_t slices, int Lq, int head_dim, bool lists, int group_rows, int64_t cus) {
  if (lists && group_rows % 256 != 0) return false;
  if (cus <= 0) return false;
  const int64_t n128 = workgroups(slices, Lq, 128), n256 = workgroups(slices, Lq, 256);
  if (n128 <= cus) return false;
  if (head_dim == 64) return n256 <= cus;
  const int64_t full = n128 / (2 * cus), rest = n128 % (2 * cus);
  const double narrow = 1.6 * full + (rest == 0 ? 0.0 : rest <= cus ? 1.0 : 1.6);
  const double wide = 1.6 * 0.95 * ((n256 + cus - 1) / cus);
  return wide < narrow;
}

// 96 rows per workgroup, three computing and four fetch waves, for dense launches of up to 32 key tiles that leave compute units
// idle as 128-row workgroups.  What is paid once per workgroup is less with fewer rows, 0.15 to 0.3 us; every tile takes 1 to 2 %
// longer, for K and V are read by a third more workgroups.  128 / 96 rows, B2 H16 d128: 576 x 700 13.83 / 13.55 us, 576 x 1500 24.15 /
// 23.89, 576 x 3000 41.84 / 41.70, but B1 H64 320 x 3000 42.4 / 42.8, x 4000 55.3 / 56.4, B1 H4 6000 x 10000 132.6 / 135.3; d64 576 x 700
// 10.92 / 10.77, x 1500 19.21 / 19.07, x 3000 33.48 / 33.64, x 4000 43.56 / 43.82, x 10000 102.2 / 103.4.
inline bool rows_of_96(int64_t slices, int Lq, int Lk, bool lists, int cus) {
  return !lists && Lk <= 2048 && workgroups(slices, Lq, 96) <= cus;
}

// Fetch-only waves beside four computing ones.  A launch of at most one 128-row workgroup per compute unit leaves half of
// the wave slots empty, and its lone waves pay for every instruction in full: 16 of the 100-odd that a wave issues per
// tile beside its MFMAs are fills.  Without / with four fetch waves, B2 H16 d128 1024 x 2521 (256 workgroups) 47.2 / 45.6 us,
// 576 x 3000 (160) 47.5 / 42.0, B1 H4 6000 x 10521 (188) 153 / 140; d64 B8 H16 256 x 680 11.8 / 11.3; lists alike (B2 H16 784 x 1924 at
// 25 % 19.2 / 17.2, 576 x 1497 15.9 / 14.5).  With a second workgroup on a compute unit there are no empty slots, and at
// head_dim 256 a wave fills its SIMD.  A workgroup with fetch waves has its compute unit to itself, so launches
// on two streams that together need more than one per compute unit no longer share any: a pair of calls, without / with,
// B1 d128 1024 x 2521: 2 x 128 workgroups 49.1 / 45.0 us, 2 x 160 (576 x 1497) 56.8 / 52.3, 2 x 192 67.1 / 68.2, 2 x 224 72.7 / 78.9,
// 2 x 256 78.9 / 88.0 (one stream 50.2 / 46.0); d64 2 x 256 49.0 / 59.0 (31.8 / 30.0).  A launch cannot know what runs beside it,
// and one stream is the usual case.
inline bool fetch_waves(int64_t slices, int Lq, int cus) { return workgroups(slices, Lq, 128) <= cus; }

// Dense attention and lists of query blocks of a multiple of 128 rows.  At head_dim 256 a wave of a 128-row workgroup fills its SIMD.
enum class BlockForm { PAIRS, WIDE, ROWS_96, FETCH, PLAIN };
inline BlockForm block_form(int64_t slices, int Lq, int Lk, int head_dim, bool lists, int group_rows, int cus) {
  if (pairs_of_waves(slices, Lq, cus)) return BlockForm::PAIRS;
  if (head_dim > 128) return BlockForm::PLAIN;
  if (wide_tiles(slices, Lq, head_dim, lists, group_rows, cus)) return BlockForm::WIDE;
  if (rows_of_96(slices, Lq, Lk, lists, cus)) return BlockForm::ROWS_96;
  return fetch_waves(slices, Lq, cus) ? BlockForm::FETCH : BlockForm::PLAIN;
}

// 192-row groups of token lists that leave compute units idle.  A group's six computing waves share four SIMDs, and the two SIMDs
// with two of them set its time.  As 64-row workgroups of pairs (pairs_of_waves), or as 96-row ones of three computing and four
// fetch waves, a computing wave has its SIMD to itself; either where every workgroup has a compute unit.  192 rows / 64 rows of
// pairs, d128 last step with 20 % of the keys, the whole step: B1 H4 64 x 64 49.3 / 32.4 us, B1 H8 40 x 40 32.0 / 18.2, B2 H4 33 x 33 at
// 5 % 22.5 / 12.5, d64 B1 H4 64 x 64 32.6 / 19.8.  192 / 96 rows: B1 H16 36 x 36 at 10 % 30.4 / 22.6, B1 H8 50 x 50 at 30 % 48.1 /
// 35.4, d64 18.8 / 15.4 and 31.1 / 23.7.
inline bool half_groups(int64_t slices, int Lq, int cus) { return workgroups(slices, Lq, 96) <= cus; }

// Token lists at head_dim 64: 192-row groups as two 3-wave workgroups (several share a compute unit, each fetches for
// itself) instead of one of 8 waves where the 8-wave workgroups leave their last round at most half
// full.  832 / 2560 keys per list, 8-wave against 3-wave: 288 groups 35.6 / - against 33.2 / - us, 384 groups 35.5 / 85.6 against 33.4 /
// 84.2, 576 groups - / 128 against - / 129; full rounds the other way (256 groups 20.7 / 44.9 against 23.2 / 52.1 us, 704 groups 53.3 /
// 127 against 56.2 / 140 us).  From the fourth round on the choice is within a few percent and stays.
inline bool three_wave_groups(int64_t slices, int Lq, int64_t cus) {
  const int64_t n = workgroups(slices, Lq, 192);
  return cus > 0 && n < 3 * cus && n % cus != 0 && 2 * (n % cus) <= cus;
}

// Token lists in groups of a multiple of 192 rows.
enum class TokenForm { PAIRS, HALF_GROUPS, THREE_WAVES, PLAIN };
inline TokenForm token_form(int64_t slices, int Lq, int head_dim, int cus) {
  if (pairs_of_waves(slices, Lq, cus)) return TokenForm::PAIRS;
  if (half_groups(slices, Lq, cus)) return TokenForm::HALF_GROUPS;
  return head_dim == 64 && three_wave_groups(slices, Lq, cus) ? TokenForm::THREE_WAVES : TokenForm::PLAIN;
}

}  // namespace lvar
