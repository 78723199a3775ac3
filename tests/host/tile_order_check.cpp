// Host-side check of the order of query tiles (lvar_amd/csrc/tile_order.h), with the arithmetic the device code uses:
//   * every query tile of every slice is taken by exactly one workgroup of the launch, and nothing else is,
//   * no XCD gets more tiles than an even split gives the fullest one,
//   * on every XCD the ragged last tiles come behind the whole ones, and the whole ones are a contiguous range,
//   * the rules that take ragged tiles out of the order, on both sides of each of their bounds,
//   * the rule that takes the instance with idle waves, likewise,
//   * the rule that orders tiles by the lengths of their lists, likewise; a slice's workgroups agree on it.
// Prints "ok <cases>" or the first violation.
#include <cstdio>
#include <vector>
#include "../../lvar_amd/csrc/tile_order.h"

using namespace lvar;

static const char* check(int slices, int nqt, bool ragged) {
  const TileOrder t = tile_order(slices, nqt, ragged);
  const int tiles = slices * nqt;
  std::vector<int> taken(tiles, 0), ranked(slices, -1);
  const int last_round = short_last_round(t, 64);
  for (int x = 0; x < TILE_XCDS; x++) {
    int here = 0, last = -1;
    bool behind = false;
    for (int i = 0; i < t.per_xcd; i++) {
      int s = -1, q = -1;
      if (!tile_of(t, i * TILE_XCDS + x, s, q)) continue;
      if (s < 0 || s >= slices || q < 0 || q >= nqt) return "tile out of range";
      taken[s * nqt + q]++;
      here++;
      if (q < t.nqt && last_round > 0) {
        const int r = ranked_slice(t, s, x, last_round);
        if (ranked[s] >= 0 && ranked[s] != r) return "workgroups of a slice that do not agree on its order";
        ranked[s] = r;
      }
      if (ragged && q == nqt - 1) { behind = true; continue; }
      if (behind) return "whole tile behind a ragged one";
      const int w = s * t.nqt + q;
      if (last >= 0 && w != last + 1) return "whole tiles of an XCD not contiguous";
      last = w;
    }
    if (here > (tiles + TILE_XCDS - 1) / TILE_XCDS) return "XCD with more tiles than an even split";
  }
  for (int n : taken)
    if (n != 1) return "tile not taken exactly once";
  return nullptr;
}

int main() {
  long cases = 0;
  for (int slices = 1; slices <= 72; slices++)
    for (int nqt = 1; nqt <= 260; nqt += nqt < 40 ? 1 : 7)
      for (int ragged = 0; ragged <= (nqt > 1 ? 1 : 0); ragged++, cases++)
        if (const char* why = check(slices, nqt, ragged != 0)) { printf("%s: %d slices of %d tiles, ragged %d\n", why, slices, nqt, ragged); return 1; }
  // one 128-row workgroup per compute unit of 256: four heads of 8065 .. 8191 rows and the like
  const int full[][2] = {{1, 256}, {2, 128}, {3, 85}, {4, 64}, {5, 51}, {9, 28}, {16, 16}, {32, 8}, {64, 4}, {128, 2}};
  for (auto& f : full)
    for (int ragged = 0; ragged <= 1; ragged++, cases++)
      if (const char* why = check(f[0], f[1], ragged != 0)) { printf("%s: %d slices of %d tiles, ragged %d\n", why, f[0], f[1], ragged); return 1; }
  // ragged tiles leave the order where they alone make the last round, with the waves of half of their rows idle
  struct { int slices, nqt, rest; bool last; } rule[] = {
      {67, 4, 30, true}, {140, 4, 96, true}, {250, 2, 96, true}, {275, 4, 30, true},
      {67, 4, 160, false}, {67, 4, 97, false},          // nearly as long as the others
      {100, 4, 30, false}, {166, 3, 30, false},         // whole tiles are left for the last round
      {32, 9, 64, false},                               // the last round holds every ragged tile
      {64, 4, 64, false}, {32, 4, 64, false}, {300, 1, 64, false}, {288, 2, 0, false}};
  for (auto& r : rule) {
    cases++;
    if (ragged_runs_last(r.slices, r.nqt, r.rest, 192, 256) != r.last) { printf("order of %d slices of %d tiles, rest %d\n", r.slices, r.nqt, r.rest); return 1; }
  }
  // block lists: heads of many tiles, more of them than compute units
  struct { int slices, nqt, rest; bool last; } lists[] = {{24, 12, 36, true}, {48, 16, 16, true}, {750, 2, 27, false}, {375, 4, 91, false}, {60, 11, 89, false},
                                                          {48, 16, 0, false}, {8, 32, 1, false}, {9, 32, 1, true}};
  for (auto& r : lists) {
    cases++;
    if (ragged_lists_last(r.slices, r.nqt, r.rest, 256) != r.last) { printf("order of %d block-list slices of %d tiles, rest %d\n", r.slices, r.nqt, r.rest); return 1; }
  }
  // idle waves: a 32nd of all, in workgroups of at least 128 rows
  struct { int waves, nqt, rest; bool pay; } idle[] = {
      {8, 7, 64, true}, {8, 2, 4, true}, {8, 4, 200, true}, {8, 18, 128, false}, {8, 18, 96, true}, {8, 7, 0, false}, {8, 2, 225, false},
      {4, 8, 60, true}, {4, 8, 96, true}, {4, 9, 96, false}, {4, 18, 64, false}, {4, 20, 4, true}, {4, 32, 4, false}, {4, 2, 97, false}, {2, 2, 20, false}};
  for (auto& r : idle) {
    cases++;
    if (idle_waves_pay(r.waves, r.nqt, r.rest) != r.pay) { printf("idle waves of %d in %d tiles per head, rest %d\n", r.waves, r.nqt, r.rest); return 1; }
  }
  // longest list first (64 places of an XCD at once): slices that reach from the rounds before into a last one of at most half of them
  struct { int slices, nqt; bool ragged; int slice, x, last_round; bool ranked; } len[] = {
      {32, 18, false, 3, 0, 64, true}, {32, 18, false, 2, 0, 64, false},      // places 54 .. 71 and 36 .. 53 of 72
      {32, 18, false, 31, 7, 64, true}, {32, 18, false, 30, 7, 64, false},
      {72, 8, false, 8, 0, 64, false}, {72, 8, false, 7, 0, 64, false},       // 64 .. 71, wholly inside the last round; 56 .. 63, up to it
      {40, 15, false, 4, 0, 64, true}, {40, 15, false, 3, 0, 64, false},      // 60 .. 74 of 75
      {20, 27, false, 2, 0, 64, false},                                       // 54 .. 80 of 68: across two XCDs
      {20, 27, false, 2, 1, 64, false}, {8, 64, false, 0, 0, 0, false},       // (seen from the other one; whole rounds)
      {32, 24, false, 2, 0, 64, true}, {32, 25, false, 2, 0, 0, false},       // last round of 32 places, of 36
      {32, 16, false, 0, 0, 0, false}, {24, 8, false, 2, 0, 0, false},        // no round before, whole rounds
      {34, 17, true, 4, 0, 64, false}, {32, 19, true, 3, 0, 64, true}};       // ragged tiles behind: 64 .. 79 of 68 whole, 54 .. 71 of 72
  for (auto& r : len) {
    cases++;
    const TileOrder t = tile_order(r.slices, r.nqt, r.ragged);
    const int last_round = short_last_round(t, 64);
    if (last_round != r.last_round || (last_round > 0 && ranked_slice(t, r.slice, r.x, last_round)) != r.ranked) {
      printf("slice %d of %d with %d tiles: last round %d, ranked %d\n", r.slice, r.slices, r.nqt, last_round, last_round > 0 && ranked_slice(t, r.slice, r.x, last_round));
      return 1;
    }
  }
  printf("ok %ld\n", cases);
  return 0;
}
