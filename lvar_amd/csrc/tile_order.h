// Order of the query tiles of a plain attention launch: which tile a workgroup takes.
//
// Workgroup ids are dealt round-robin to the 8 XCDs, each with an L2 of its own, so an XCD takes a contiguous range of
// (batch, head, query tile) and the K/V of one head stay in its L2.  Ragged last tiles may be taken out of that order and
// run behind the whole ones of their XCD.  Every XCD gets the same number of places for whole and ragged tiles together:
// with a share of each rounded up on its own, 252 whole and 4 ragged tiles put 33 workgroups on the 32 compute units of four
// XCDs, and where a workgroup fills a compute unit that is a second round (B1 H4 d128 8100 x 8100: 222 us, 128 us with
// even places; H9 3500 rows 220, 126).  Integer arithmetic shared by the device code and by a host-side test.
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

constexpr int TILE_XCDS = 8;

struct TileOrder {
  int nqt;            // query tiles of a (batch, head) that run in order: all of them, or all but the ragged last one
  int whole;          // how many these are over all slices
  int whole_per_xcd;  // how many of them an XCD takes at most
  int ragged;         // ragged last tiles that run behind them: one per slice, or none
  int per_xcd;        // places per XCD; the launch has TILE_XCDS * per_xcd workgroups
};

LVAR_HD TileOrder tile_order(int slices, int nqt, bool ragged_last) {
  TileOrder t;
  t.nqt = ragged_last ? nqt - 1 : nqt;
  t.whole = slices * t.nqt;
  t.whole_per_xcd = (t.whole + TILE_XCDS - 1) / TILE_XCDS;
  t.ragged = ragged_last ? slices : 0;
  t.per_xcd = (t.whole + t.ragged + TILE_XCDS - 1) / TILE_XCDS;
  return t;
}

// Tile of workgroup `id`: slice and query tile, or false where there is none.  The places that the whole tiles leave on
// XCD x go to ragged ones, in slice order.
LVAR_HD bool tile_of(const TileOrder& t, unsigned id, int& slice, int& qt) {
  const int x = (int)(id % TILE_XCDS), i = (int)(id / TILE_XCDS);
  const int first = x * t.whole_per_xcd < t.whole ? x * t.whole_per_xcd : t.whole;   // whole tiles of the XCDs before x
  const int mine = t.whole - first < t.whole_per_xcd ? t.whole - first : t.whole_per_xcd;
  if (i < mine) {
    slice = (first + i) / t.nqt;
    qt = first + i - slice * t.nqt;
    return true;
  }
  slice = x * t.per_xcd - first + (i - mine);
  qt = t.nqt;
  return i < t.per_xcd && slice < t.ragged;
}

// The place of an XCD at which a last round of at most half of its places begins, or 0 where a launch ends otherwise.  `round_places`:
// places of an XCD that run at once.
LVAR_HD int short_last_round(const TileOrder& t, int round_places) {
  if (round_places <= 0) return 0;
  const int full = t.per_xcd / round_places * round_places;   // places before the last round
  return full < t.per_xcd && 2 * (t.per_xcd - full) <= round_places ? full : 0;
}

// Whether the tiles of a slice, one of which runs on XCD x, run longest list first: slices that lie in that XCD and reach from the
// rounds before into a short last one (its place from short_last_round), so that what starts late is short.  The others keep their
// order: a ranked tile waits for the lengths of its slice's lists before its own list is read, and where a whole slice starts in the
// last round that wait is all that would come of it (ranked / not, B3 H24 900 x 2000 at 30 % 38.6 / 37.6 us, B1 H300 256 x 4000 at 10 %
// 34.2 / 33.0).  Natural order / longest first, d128, 128-row tiles, two per compute unit: random lists B2 H16 48 x 48 (576 tiles on
// 512 places) at 25 % 80.7 / 74.6 us, at 10 % 43.1 / 39.0, B2 H20 44 x 44 78.7 / 78.4 and 45.1 / 41.5; sink + window 48 x 48 57.7 / 55.3,
// B2 H12 56 x 56 82.9 / 81.7; best-scoring blocks, nearly of one length, 48 x 48 25 % 72.6 / 72.7, 10 % 64.2 / 63.3; lists of exactly
// one length lose the wait, 0.3 us.  With ragged tiles behind the whole ones it is the draw: B1 H24 56 x 56 115.0 / 118.4 and 56.4 /
// 56.3, lists of a few entries (48 heads 1600 x 4121, 5 % of the 128-key blocks, eight draws) -5 .. +8 %.
// With the last round 46 / 64 full random lists lose 1.8 %.  head_dim 64 loses 1 % (a third workgroup per compute unit covers the
// end), 64-row tiles gain nothing.
LVAR_HD bool ranked_slice(const TileOrder& t, int slice, int x, int last_round) {
  const int first = slice * t.nqt - x * t.whole_per_xcd, last = first + t.nqt - 1;   // places on XCD x
  return first >= 0 && first < last_round && last >= last_round && last < t.whole_per_xcd;
}

// Whether the ragged last tiles of token lists with fetch-only waves (one workgroup per compute unit) run behind the whole
// ones.  The waves without rows do not compute, so with at least half of them idle such a tile is the shorter workgroup, and
// it pays where the launch can end on a round of nothing else, with every whole tile in the full rounds before it.  832 of
// 4121 keys, d128, 192-row groups with 30 rows in the last one, behind against in order: 67 heads of 4 tiles on 256 compute
// units -20 %, 140 heads -8 %, 275 -3 %; where whole tiles are left for the last round +2 .. +4 % (100 heads of 4, 166 of 3).
LVAR_HD bool ragged_runs_last(int slices, int nqt, int rest, int rows, int cus) {
  if (cus <= 0 || nqt < 2 || rest == 0 || 2 * rest > rows) return false;
  const int total = slices * nqt, left = total % cus;
  return total > cus && left > 0 && left < slices;
}

// The same for block lists.  The last tile of a grid has the shorter lists of a sink + window mask (50 drawn layers of at
// least 12 tiles per head: -0.7 % on average, -5.6 .. +3.7 %), and lists of a score or of random length come out even, while
// its second visit to the K/V of a head costs the more the fewer tiles share it: in order / behind, 25 % of 4121 keys, d128,
// 1500 tiles in heads of 2 170 / 190 us, of 4 152 / 161, of 8 139 / 140.  Dense attention gains nothing from it at any size
// (2 tiles 71 / 80 us; d256, 3 tiles 436 / 487).
LVAR_HD bool ragged_lists_last(int slices, int nqt, int rest, int cus) { return rest != 0 && nqt >= 12 && slices * nqt > cus; }

// Whether an instance is taken whose waves without rows do not compute, in dense and block-list launches of workgroups
// where no wave only fetches: a second loop in the kernel costs every workgroup up to a percent, and a last tile has only so
// many idle waves; what they save is matrix instructions, and so power, in launches that run long enough for the clock to
// follow.  d128, with it against without, kept up for 150 ms each: dense 128-row workgroups with 3 of 8 waves of a head idle
// -3 .. -12 %, 2 of 32 -0.4 .. -3 %, 2 of 64 -0.2 .. -0.6 %; lists of 25 % with 3 of 16 -1 .. -5 %, 3 of 48 -0.4 .. -3 %, 3 of
// 80 +0.1 .. -2.5 %, 2 of 80 +0.6 .. -0.5 %, 1 of 80 +1.6 .. -0.1 %; 256-row ones with 6 of 56 111.7 / 106.5 us, 4 of 144 -0.4 %,
// 2 of 144 nothing.  64-row workgroups lose up to 1 % at any share.
LVAR_HD bool idle_waves_pay(int waves, int nqt, int rest) {
  const int idle = rest == 0 ? 0 : waves - (rest + 31) / 32;
  return waves >= 4 && idle > 0 && 32 * idle >= waves * nqt;
}

}  // namespace lvar
