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

}  // namespace lvar
