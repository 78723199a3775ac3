// Host-side check of the rules that choose the form of a plain attention launch (lvar_amd/csrc/launch_forms.h), on a chip of 256
// compute units and on both sides of each bound.  Prints "ok <cases>" or the first violation.
#include <cstdio>
#include "../../lvar_amd/csrc/launch_forms.h"

using namespace lvar;

int main() {
  int cases = 0;
  struct { int slices, Lq, Lk, d; bool lists; int group_rows; BlockForm form; } block[] = {
      {256, 64, 64, 128, false, 128, BlockForm::PAIRS}, {256, 65, 64, 128, false, 128, BlockForm::ROWS_96},   // 256 64-row workgroups, 512
      {4, 4096, 10521, 64, false, 128, BlockForm::PAIRS}, {4, 4097, 1000, 64, false, 128, BlockForm::ROWS_96},
      {32, 512, 1000, 256, true, 128, BlockForm::PAIRS}, {32, 513, 1000, 256, true, 128, BlockForm::PLAIN},
      {8, 2048, 64, 128, true, 256, BlockForm::PAIRS}, {257, 1, 1, 128, false, 128, BlockForm::PLAIN},
      {32, 576, 2048, 128, false, 128, BlockForm::ROWS_96}, {32, 576, 2049, 128, false, 128, BlockForm::FETCH},   // 32 key tiles
      {32, 576, 2048, 128, true, 128, BlockForm::FETCH},                                                      // lists have no rows of 96
      {256, 96, 500, 64, false, 128, BlockForm::ROWS_96}, {256, 97, 500, 64, false, 128, BlockForm::FETCH},   // 256 96-row workgroups, 512
      {256, 128, 500, 64, false, 128, BlockForm::FETCH}, {256, 129, 500, 64, false, 128, BlockForm::WIDE},    // 256 128-row ones, 512 (256 of 256 rows)
      {257, 128, 500, 64, false, 128, BlockForm::PLAIN}, {513, 100, 500, 64, false, 128, BlockForm::PLAIN},
      {32, 4096, 10521, 128, false, 128, BlockForm::WIDE}, {32, 4096, 10521, 64, false, 128, BlockForm::PLAIN},
      {32, 4096, 10521, 128, true, 128, BlockForm::PLAIN}, {32, 4096, 10521, 128, true, 256, BlockForm::WIDE},
      {32, 4096, 10521, 256, false, 128, BlockForm::PLAIN}, {96, 1024, 2521, 128, false, 128, BlockForm::PLAIN},
      {97, 1024, 2521, 128, false, 128, BlockForm::WIDE}, {36, 1024, 2521, 128, true, 128, BlockForm::PLAIN},
      {36, 1024, 2521, 128, true, 256, BlockForm::WIDE}};
  for (auto& r : block) {
    cases++;
    const BlockForm f = block_form(r.slices, r.Lq, r.Lk, r.d, r.lists, r.group_rows, 256);
    if (f != r.form) { printf("form %d of %d slices %d x %d, head_dim %d, lists %d of %d rows\n", (int)f, r.slices, r.Lq, r.Lk, r.d, r.lists, r.group_rows); return 1; }
  }
  struct { int slices, Lq, d; TokenForm form; } token[] = {
      {4, 4096, 128, TokenForm::PAIRS}, {4, 4097, 128, TokenForm::HALF_GROUPS}, {4, 6144, 128, TokenForm::HALF_GROUPS},
      {4, 6145, 128, TokenForm::PLAIN}, {256, 64, 64, TokenForm::PAIRS}, {256, 65, 64, TokenForm::HALF_GROUPS},
      {256, 97, 64, TokenForm::PLAIN},                                                  // 256 groups: a full round
      {257, 97, 64, TokenForm::THREE_WAVES}, {257, 97, 128, TokenForm::PLAIN}, {384, 192, 64, TokenForm::THREE_WAVES},
      {385, 192, 64, TokenForm::PLAIN}, {129, 192, 64, TokenForm::PLAIN}, {128, 192, 64, TokenForm::HALF_GROUPS},
      {640, 192, 64, TokenForm::THREE_WAVES}, {641, 192, 64, TokenForm::PLAIN}, {769, 192, 64, TokenForm::PLAIN}};
  for (auto& r : token) {
    cases++;
    const TokenForm f = token_form(r.slices, r.Lq, r.d, 256);
    if (f != r.form) { printf("form %d of token lists, %d slices of %d rows, head_dim %d\n", (int)f, r.slices, r.Lq, r.d); return 1; }
  }
  // no compute unit known: the plain launch
  if (block_form(4, 100, 100, 128, false, 128, 0) != BlockForm::PLAIN || token_form(4, 100, 64, 0) != TokenForm::PLAIN) { printf("no compute units\n"); return 1; }
  printf("ok %d\n", cases);
  return 0;
}
