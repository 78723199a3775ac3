// Block-list build on the GPU: per (batch, head, query block) row, keep the always-on blocks of a
// static base mask plus the best-scoring remaining blocks up to a target count, and emit the
// compacted ascending block list (flex BlockMask layout: count + indices, unused tail zero).
//
// One wave per row, the keys of the row in registers (KPL per lane, block c * 64 + lane): no LDS, no barrier.  Selection
// is by exact rank: block j is kept if fewer than `extra` non-base blocks beat it, where "beats" is (score greater) or
// (score equal and index smaller), i.e. the order of a stable descending sort, so the result is a pure function of the
// scores.  The cut is found by bisecting the 32-bit sort key: a step is one compare and one population count per 64
// blocks, and the search ends as soon as exactly `extra` keys reach the trial value.  (Counting the keys above every
// key, as one 256-thread workgroup per row, is quadratic: 39 us for 6144 rows x 256 blocks and 6.2 us for 576 x 101
// against 14 and 4.9 us.)
#include "common.h"
#include "launch.h"

namespace lvar {

constexpr int MASKLIST_MAX_NK = 2048;  // blocks per row held in registers
constexpr int MASKLIST_NT = 256;       // four rows

template <int KPL>
__global__ __launch_bounds__(MASKLIST_NT) void block_topk_lists_kernel(const MaskListParams p) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // (b*H + h)*nQ + i
  if (row >= p.rows) return;
  const int nK = p.nK;
  const float* s = p.scores + (int64_t)row * nK;
  const uint8_t* base = p.base ? p.base + (int64_t)(row % p.nQ) * nK : nullptr;

  // keys: 0 for base blocks and behind the end, real keys are larger
  float x[KPL];
  bool isb[KPL];
#pragma unroll
  for (int c = 0; c < KPL; c++) {
    const int j = min(c * 64 + lane, nK - 1);   // (clamped: the loads go out together)
    x[c] = s[j];
    isb[c] = base ? base[j] != 0 : false;
  }
  uint32_t key[KPL];
  int nbase = 0;
#pragma unroll
  for (int c = 0; c < KPL; c++) {
    const bool in = c * 64 + lane < nK;
    isb[c] = isb[c] && in;
    key[c] = in && !isb[c] ? real_key(x[c]) : 0u;
    nbase += __builtin_popcountll(__builtin_amdgcn_ballot_w64(isb[c]));
  }
  const int extra = max(0, min(p.target, nK) - nbase);
  auto count = [&](uint32_t v) {
    int n = 0;
#pragma unroll
    for (int c = 0; c < KPL; c++) n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(key[c] >= v));
    return n;
  };
  // kept: keys above `cut` and the first `ties` equal to it
  uint32_t cut = 0u;
  int ties = 0;
  if (extra == 0) {
    cut = 0xffffffffu;
  } else if (extra < nK - nbase) {
    int n = 0;
    for (int bit = 31; bit >= 0; bit--) {
      const uint32_t v = cut | (1u << bit);
      const int m = count(v);
      if (m < extra) continue;
      cut = v;
      n = m;
      if (m == extra) break;
    }
    if (n == extra) cut--;                       // every key that reaches the trial value
    else ties = extra - (cut == 0xffffffffu ? 0 : count(cut + 1u));
  }

  int32_t* out = p.kv_indices + (int64_t)row * nK;
  int written = 0;
#pragma unroll
  for (int c = 0; c < KPL; c++) {
    bool keep = isb[c] || key[c] > cut;
    if (ties > 0) {
      const unsigned long long eq = __builtin_amdgcn_ballot_w64(key[c] == cut);
      if (key[c] == cut && __builtin_popcountll(eq & ((1ull << lane) - 1ull)) < ties) keep = true;
      ties = max(0, ties - __builtin_popcountll(eq));
    }
    const unsigned long long bal = __builtin_amdgcn_ballot_w64(keep);
    if (keep) out[written + __builtin_popcountll(bal & ((1ull << lane) - 1ull))] = c * 64 + lane;
    written += __builtin_popcountll(bal);
  }
  for (int t = written + lane; t < nK; t += 64) out[t] = 0;
  if (lane == 0) p.kv_num_blocks[row] = written;
}

template <int KPL>
static bool block_topk_try(const MaskListParams& p, hipStream_t stream) {
  if (p.nK > 64 * KPL) return false;
  hipLaunchKernelGGL(block_topk_lists_kernel<KPL>, dim3((p.rows + 3) / 4), dim3(MASKLIST_NT), 0, stream, p);
  return true;
}

int launch_block_topk_lists(const MaskListParams& p, hipStream_t stream) {
  if (p.nK > MASKLIST_MAX_NK) return LVAR_EUNSUPPORTED;
  block_topk_try<1>(p, stream) || block_topk_try<2>(p, stream) || block_topk_try<3>(p, stream) || block_topk_try<4>(p, stream) ||
      block_topk_try<6>(p, stream) || block_topk_try<8>(p, stream) || block_topk_try<12>(p, stream) || block_topk_try<16>(p, stream) ||
      block_topk_try<24>(p, stream) || block_topk_try<32>(p, stream);
  return hipGetLastError() == hipSuccess ? LVAR_OK : LVAR_ELAUNCH;
}

}  // namespace lvar
