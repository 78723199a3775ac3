// Key-list build on the GPU for the token-list attention path: exact per-row top-k selection of the
// column sums, the cross-scale query-group remap fused with the local-run append, and the
// compaction of a boolean mask into index lists.  All three are HBM/L2-bound integer work: one pass
// (or a few L2-resident passes) over the rows, ballot/prefix compaction, no sorting.
#include <utility>
#include "common.h"
#include "launch.h"
#include "score_bins.h"

namespace lvar {

__device__ __forceinline__ int lanes_below(unsigned long long bal, int lane) {
  return __builtin_popcountll(bal & ((1ull << lane) - 1ull));
}

// Inclusive scan over the 64 lanes of a wave with data-parallel-primitive moves (row shifts by 1, 2, 4, 8 inside the rows
// of 16 lanes, then the last lane of row 0 / 2 broadcast into row 1 / 3 and the last lane of row 1 into rows 2 and 3):
// six dependent vector instructions instead of six round trips through the LDS crossbar.  Lanes that a move does not
// reach take the identity.  Lane 63 ends up with the reduction over the wave.
template <class Op>
__device__ __forceinline__ int wave_scan(int v, const int identity, Op op) {
  v = op(v, __builtin_amdgcn_update_dpp(identity, v, 0x111, 0xf, 0xf, false));   // row_shr:1
  v = op(v, __builtin_amdgcn_update_dpp(identity, v, 0x112, 0xf, 0xf, false));   // row_shr:2
  v = op(v, __builtin_amdgcn_update_dpp(identity, v, 0x114, 0xf, 0xf, false));   // row_shr:4
  v = op(v, __builtin_amdgcn_update_dpp(identity, v, 0x118, 0xf, 0xf, false));   // row_shr:8
  v = op(v, __builtin_amdgcn_update_dpp(identity, v, 0x142, 0xa, 0xf, false));   // row_bcast:15 into rows 1 and 3
  v = op(v, __builtin_amdgcn_update_dpp(identity, v, 0x143, 0xc, 0xf, false));   // row_bcast:31 into rows 2 and 3
  return v;
}
__device__ __forceinline__ uint32_t wave_umax(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_readlane(wave_scan((int)v, 0, [](int a, int b) { return (int)max((uint32_t)a, (uint32_t)b); }), 63);
}
__device__ __forceinline__ uint32_t wave_umin(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_readlane(wave_scan((int)v, -1, [](int a, int b) { return (int)min((uint32_t)a, (uint32_t)b); }), 63);
}
// Smallest value of each aligned group of G lanes (2, 4 or 8; ~0 does not count), over the groups of the wave the largest (0: none)
template <int G>
__device__ __forceinline__ uint32_t wave_max_of_group_min(uint32_t v) {
  auto mv = [](uint32_t x, auto ctrl) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, decltype(ctrl)::value, 0xf, 0xf, true); };
  auto close = [&](auto last) { if constexpr (decltype(last)::value) v = v == 0xffffffffu ? 0u : v; };
  uint32_t o = mv(v, std::integral_constant<int, 0xB1>{});    // quad_perm: neighbours
  v = min(v, o);
  close(std::bool_constant<G == 2>{});
  o = mv(v, std::integral_constant<int, 0x4E>{});             // quad_perm: pairs
  v = G >= 4 ? min(v, o) : max(v, o);
  close(std::bool_constant<G == 4>{});
  o = mv(v, std::integral_constant<int, 0x141>{});            // row_half_mirror: fours
  v = G >= 8 ? min(v, o) : max(v, o);
  close(std::bool_constant<G == 8>{});
  v = max(v, mv(v, std::integral_constant<int, 0x140>{}));    // row_mirror: eights
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));   // row_bcast:15 into rows 1 and 3
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));   // row_bcast:31 into rows 2 and 3
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
// Reduction over each row of 16 lanes, in all of them
template <class Op, class T>
__device__ __forceinline__ void row_all(Op op, T& v) {
  auto mv = [](T x, auto ctrl) { return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, true)); };
  v = op(v, mv(v, std::integral_constant<int, 0xB1>{}));    // quad_perm: neighbours
  v = op(v, mv(v, std::integral_constant<int, 0x4E>{}));    // quad_perm: pairs
  v = op(v, mv(v, std::integral_constant<int, 0x141>{}));   // row_half_mirror: fours
  v = op(v, mv(v, std::integral_constant<int, 0x140>{}));   // row_mirror: eights
}

// ---------------------------------------------------------------------------------------------
// Exact top-k per row by radix select.  One 512-thread workgroup per row; wave w owns the w-th
// contiguous eighth of the (padded) row and every thread keeps its KPT keys in registers (KPT = 0:
// rows too long for that are re-read from L2 in every pass).
//   a histogram pass (11 bits, starting below the bits that all keys of the row share; LDS atomics)
//   finds the bin of the k-th largest key; the keys of that bin are compared with each other directly
//   (or, if they are too many, go through up to two more histogram passes), which gives the exact
//   value T of the k-th largest key and the number `need` of keys equal to T that belong to the
//   selection (ties go to the smaller column);
//   a counting pass gives every wave its number of selected keys, the last pass writes the selected
//   columns in ascending order (ballot compaction into an LDS ring, full-width stores).
// ---------------------------------------------------------------------------------------------
constexpr int TOPK_BINS = SCORE_BINS;
constexpr int TOPK_SHARED_MAX_N = 12288;   // longest row of 1024 threads where two rows share a compute unit
constexpr int TOPK_CAND = 256;   // keys of the first pass's bin that are resolved by direct comparison

// UNION: the output row is the ascending merge of the selection with the row's own list of W columns (in any order,
// columns that are listed or selected several times come out as often), as int64.  How often each column is listed sits
// in LDS as 16-bit counts, so a column's place in the merge is one more term of the scan that places the selection.
template <int KPT, int NT, bool UNION>
__global__ __launch_bounds__(NT, (KPT >= 1 && KPT <= 24) ? (NT == 512 ? 6 : 4) : 1) void topk_token_lists_kernel(const TopkListParams p) {
  constexpr int NW = NT / 64;
  extern __shared__ uint32_t listed[];   // UNION: two 16-bit counts per word
  __shared__ int hist[TOPK_BINS];
  __shared__ __attribute__((aligned(16))) uint32_t cand[TOPK_CAND];
  __shared__ int wsum[NW];
  __shared__ int sel[2];  // chosen bin, keys still wanted inside it
  __shared__ int ncand;
  __shared__ int wgt[NW], weq[NW];
  const int row = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* s = p.scores + (int64_t)row * p.score_stride;
  int32_t* out = p.indices + (int64_t)row * p.out_stride;
  const int n = p.n;
  int want = min(max(p.k, 0), n);  // keys still to be found among those matching the prefix
  if (tid == 0 && p.counts) p.counts[row] = want;
  // columns [k, zero_to) of the list row: defined (zero) instead of whatever the buffer held
  for (int t = want + tid; t < p.zero_to; t += NT) out[t] = 0;
  if (want == 0) return;
  if constexpr (UNION)
    for (int t = tid; t < TOPK_BINS; t += NT) hist[t] = 0;
  int64_t more_first = 0;   // this thread's first entry of the row's own list, requested ahead of the scores
  if constexpr (UNION) {
    if (tid < p.W) more_first = p.more[(int64_t)row * p.W + tid];
    for (int t = tid; t < (n + 1) / 2; t += NT) listed[t] = 0u;
  }

  // chunk c of wave w covers columns (w * cpw + c) * 64 .. +63
  const int cpw = KPT ? KPT : ((n + NT - 1) / NT);
  const int col0 = wave * cpw * 64 + lane;
  uint32_t keys[KPT ? KPT : 1];
  uint32_t kmax = 0u, kmin = 0xffffffffu;   // over the real columns of this thread
  if (KPT) {
    // All KPT loads are issued back to back (a branch around each would make them KPT dependent round trips):
    // buffer loads bounded to the row, so that columns beyond n read as zero instead of reaching past the row.
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)s, 0, n * 4, 0x00020000);
    uint32_t raw[KPT ? KPT : 1];
#pragma unroll
    for (int c = 0; c < KPT; c++) raw[c] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, col0 * 4, c * 256, 0);
#pragma unroll
    for (int c = 0; c < KPT; c++) {
      const bool real = col0 + c * 64 < n;
      keys[c] = real ? real_key(__builtin_bit_cast(float, raw[c])) : 0u;
      kmax = max(kmax, keys[c]);
      kmin = min(kmin, real && (!UNION || keys[c] > KEY_NEG_INF) ? keys[c] : 0xffffffffu);
    }
  } else {
    for (int c = 0; c < cpw; c++) {
      const int j = col0 + c * 64;
      if (j < n) { const uint32_t key = real_key(s[j]); kmax = max(kmax, key); kmin = min(kmin, key); }
    }
  }
  // visit(f): f(column, key) for every chunk of this wave (all 64 lanes call it together); padding columns have key 0.
  // The column numbers are formed from a copy of col0 that the compiler cannot relate to the ones of the loads:
  // kept alive from there they would be spilled, and their reloads would wait for every store in flight.
  int c0 = col0;
  asm volatile("" : "+v"(c0));
  auto visit = [&](auto&& f) {
    if (KPT) {
#pragma unroll
      for (int c = 0; c < KPT; c++) f(c0 + c * 64, keys[c]);
    } else {
      for (int c = 0; c < cpw; c++) {
        const int j = c0 + c * 64;
        f(j, (j < n) ? real_key(s[j]) : 0u);
      }
    }
  };

  // Column sums of one row sit in a narrow range: with the digits taken from the top of the key nearly every key
  // would fall into a handful of bins of the first pass and the LDS atomics of a wave would serialise on them.  The
  // bits that the largest and the smallest key of the row have in common are therefore taken as known, and the
  // digits start at the first bit in which keys differ: `top` low bits are left to resolve, 11 at a time.
  if constexpr (UNION) {
    // the bulk of the row, see score_bins.h (threads without a score stay out of it)
    constexpr int G = score_group(KPT);
    const bool any = kmin <= kmax;
    kmax = wave_max_of_group_min<G>(any ? kmax : 0xffffffffu);
    kmin = ~wave_max_of_group_min<G>(any ? ~kmin : 0xffffffffu);
  } else {
    kmax = wave_umax(kmax);
    kmin = wave_umin(kmin);
  }
  if (lane == 0) { wgt[wave] = (int)kmax; weq[wave] = (int)kmin; }
  if (tid == 0) ncand = 0;
  __syncthreads();
  float narrow = 0.f;   // UNION: width of the narrowest bulk of a wave
  if constexpr (UNION) {
    static_assert(NW == 16, "one wave per lane of a row of 16");
    kmax = (uint32_t)wgt[lane & 15];
    kmin = (uint32_t)weq[lane & 15];
    const float width = score_width(kmin, kmax);
    narrow = width > 0.f && ((lane & 15) + 1) * KPT * 64 <= n ? width : INFINITY;   // (the last wave's may be that of a few columns)
    row_all([](uint32_t a, uint32_t b) { return max(a, b); }, kmax);
    row_all([](uint32_t a, uint32_t b) { return min(a, b); }, kmin);
    row_all([](float a, float b) { return fminf(a, b); }, narrow);
    kmax = __builtin_amdgcn_readfirstlane(kmax);
    kmin = __builtin_amdgcn_readfirstlane(kmin);
  } else {
#pragma unroll
    for (int w = 0; w < NW; w++) { kmax = max(kmax, (uint32_t)wgt[w]); kmin = min(kmin, (uint32_t)weq[w]); }
  }
  if constexpr (UNION) {   // (read behind at least one more barrier)
    const int64_t* more = p.more + (int64_t)row * p.W;
    for (int t = tid; t < p.W; t += NT) {
      const int j = (int)max((int64_t)0, min((int64_t)n - 1, t < NT ? more_first : more[t]));
      atomicAdd(&listed[j >> 1], 1u << (16 * (j & 1)));
    }
  }
  // bits that keys of [lo, hi] need not share
  auto differing = [](uint32_t lo, uint32_t hi) { return 32 - __builtin_clz((hi ^ lo) | 1u) + (((hi ^ lo) == 0u) ? -1 : 0); };   // 0 when all keys are equal
  auto above_bits = [](int bits) -> uint32_t { return bits >= 32 ? 0u : ~((1u << bits) - 1u); };
  // (UNION: its range is not that of all keys, so nothing is known from it)
  int top = UNION ? 32 : differing(kmin, kmax);
  uint32_t pmask = above_bits(top);
  uint32_t prefix = kmax & pmask;
  // UNION, first pass: bins of equal width.  Where that of the threshold is too full after all, the passes by digits follow
  // over its keys, [klo, khi].
  int bin[UNION ? KPT : 1], lbin = 0;
  uint32_t klo = 0u, khi = 0xffffffffu;
  auto in_play = [&](uint32_t key) -> bool { return (key & pmask) == prefix && (!UNION || (klo <= key && key <= khi)); };
  // One more key in bin `at`, for the lanes that ask.  UNION, whose digits are a second choice where keys crowd: the lanes that
  // share the bin of the first one count at once, not one after the other (99 % equal scores 40 -> 21 us).
  auto tally = [&](int at, bool counts) {
    if constexpr (UNION) {
      const unsigned long long asked = __builtin_amdgcn_ballot_w64(counts);
      if (asked == 0ull) return;
      const int first = __builtin_ctzll(asked);
      const int b0 = __builtin_amdgcn_readlane(at, first);
      const unsigned long long same = __builtin_amdgcn_ballot_w64(counts && at == b0);
      if (__builtin_popcountll(same) > 8) {
        if (lane == first) atomicAdd(&hist[b0], __builtin_popcountll(same));
        counts = counts && at != b0;
      }
    }
    if (counts) atomicAdd(&hist[at], 1);
  };
  using yes = std::true_type;
  using no = std::false_type;
  // The bin that holds the want-th key from the top, and how many of its keys are wanted: thread t owns the bpt bins
  // nbins-1 - t*bpt .. (descending).
  auto find_bin = [&](int nbins) {
    const int bpt = (nbins + NT - 1) / NT;   // 1 when there are as many threads as bins (then every thread owns one)
    const int btop = nbins - 1 - tid * bpt;
    int mine = 0;
    for (int e = 0; e < bpt; e++) mine += (btop - e >= 0) ? hist[btop - e] : 0;
    const int incl = wave_scan(mine, 0, [](int a, int b) { return a + b; });
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int before = incl - mine;
    for (int w = 0; w < wave; w++) before += wsum[w];
    if (before < want && want <= before + mine) {  // exactly one thread
      int acc = before, bin = btop;
      for (int e = 0; e < bpt; e++) {
        const int h = (btop - e >= 0) ? hist[btop - e] : 0;
        if (acc + h >= want) { bin = btop - e; break; }
        acc += h;
      }
      sel[0] = bin;
      sel[1] = want - acc;
    }
    __syncthreads();
    want = sel[1];
    // (the next write of `sel` lies behind three more barriers: no barrier needed after these reads)
  };
  // After the first pass the chosen bin usually holds a few dozen keys.  They are copied to LDS, and if they
  // fit, every one of them counts the candidates above it: the one with fewer than `want` above and at least
  // `want` at or above is the threshold, and the other passes are not needed.
  auto resolve = [&](auto by_bin) -> bool {
    int c = 0;
    visit([&](int j, uint32_t key) {
      bool m;
      if constexpr (decltype(by_bin)::value) m = bin[c++] == lbin;
      else m = in_play(key);
      const unsigned long long bm = __builtin_amdgcn_ballot_w64(m);
      if (bm != 0ull) {
        int base = 0;
        if (lane == 0) base = atomicAdd(&ncand, __builtin_popcountll(bm));
        base = __builtin_amdgcn_readfirstlane(base);
        const int at = base + lanes_below(bm, lane);
        if (m && at < TOPK_CAND) cand[at] = key;
      }
    });
    __syncthreads();
    const int nc = ncand;
    if (nc > TOPK_CAND) return false;
    if (tid < nc) {
      const uint32_t kt = cand[tid];
      int above = 0, at_or_above = 0;
      // four candidates per LDS read (all lanes read the same address): the loop is bound by the latency of its reads
      for (int u = 0; u < nc; u += 4) {
        const u32x4 ku = *(const u32x4*)(cand + u);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const bool in = u + e < nc;
          above += in && ku[e] > kt;
          at_or_above += in && ku[e] >= kt;
        }
      }
      if (above < want && want <= at_or_above) { sel[0] = (int)kt; sel[1] = want - above; }   // equal keys write equal values
    }
    __syncthreads();
    prefix = (uint32_t)sel[0];
    want = sel[1];
    return true;
  };
  bool found = false, first = true;
  if constexpr (UNION) {
    ScoreBins bins;
    if (score_bins(kmin, kmax, narrow, bins)) {
#pragma unroll
      for (int c = 0; c < KPT; c++) bin[c] = score_bin(bins, keys[c]);
#pragma unroll
      for (int c = 0; c < KPT; c++) atomicAdd(&hist[bin[c]], 1);
      __syncthreads();
      find_bin(TOPK_BINS);
      lbin = sel[0];
      found = resolve(yes{});
      if (!found) {
        uint32_t hi = 0u, lo = 0xffffffffu;
#pragma unroll
        for (int c = 0; c < KPT; c++)
          if (bin[c] == lbin) { hi = max(hi, keys[c]); lo = min(lo, keys[c]); }
        hi = wave_umax(hi);
        lo = wave_umin(lo);
        if (lane == 0) { wgt[wave] = (int)hi; weq[wave] = (int)lo; }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < NW; w++) { hi = max(hi, (uint32_t)wgt[w]); lo = min(lo, (uint32_t)weq[w]); }
        if (tid == 0) ncand = 0;   // (every wave has read it ahead of that barrier)
        klo = lo;
        khi = hi;
        top = differing(klo, khi);
        pmask = above_bits(top);
        prefix = khi & pmask;
      }
    }
  }
  if (top == 0) __syncthreads();   // no pass below to separate these reads of wgt / weq from their reuse
  for (int hi = found ? 0 : top; hi > 0;) {
    const int shift = max(0, hi - 11);
    const int bits = hi - shift;
    hi = shift;
    const int nbins = 1 << bits;
    for (int t = tid; t < nbins; t += NT) hist[t] = 0;
    __syncthreads();
    visit([&](int j, uint32_t key) {
      tally((key >> shift) & (nbins - 1), in_play(key));
    });
    __syncthreads();
    find_bin(nbins);
    prefix |= (uint32_t)sel[0] << shift;
    pmask |= (uint32_t)(nbins - 1) << shift;
    if (first && hi > 0) {
      first = false;
      if (resolve(no{})) break;
    }
  }
  const uint32_t T = prefix;  // key of the k-th largest element
  const int need = want;      // selected keys equal to T (the first `need` of them by column)

  int gt = 0, eq = 0, times = 0;
  const uint16_t* listed16 = (const uint16_t*)listed;
  visit([&](int j, uint32_t key) {
    gt += __builtin_popcountll(__builtin_amdgcn_ballot_w64(key > T));
    eq += __builtin_popcountll(__builtin_amdgcn_ballot_w64(key == T));
    if constexpr (UNION) times += j < n ? (int)listed16[j] : 0;
  });
  if constexpr (UNION) gt += __builtin_amdgcn_readlane(wave_scan(times, 0, [](int a, int b) { return a + b; }), 63);
  if (lane == 0) { wgt[wave] = gt; weq[wave] = eq; }
  __syncthreads();
  int pos = 0, eq_before = 0;
  for (int w = 0; w < wave; w++) {
    pos += wgt[w] + max(0, min(weq[w], need - eq_before));
    eq_before += weq[w];
  }
  int eq_left = max(0, need - eq_before);
  if constexpr (UNION) {
    int64_t* out64 = p.out64 + (int64_t)row * p.out_stride;
    visit([&](int j, uint32_t key) {
      unsigned long long bk = __builtin_amdgcn_ballot_w64(key > T);
      const unsigned long long beq = __builtin_amdgcn_ballot_w64(key == T);
      if (beq != 0ull && eq_left > 0) {
        bk |= __builtin_amdgcn_ballot_w64(key == T && lanes_below(beq, lane) < eq_left);
        eq_left = max(0, eq_left - __builtin_popcountll(beq));
      }
      const int mult = j < n ? (int)listed16[j] : 0;
      const int mine = (int)((bk >> lane) & 1ull) + mult;
      if (__builtin_amdgcn_ballot_w64(mine > 1) == 0ull) {
        // (the usual case: listed columns are listed once and not selected)
        bk = __builtin_amdgcn_ballot_w64(mine > 0);
        if (mine) out64[pos + lanes_below(bk, lane)] = j;
        pos += __builtin_popcountll(bk);
      } else {
        const int incl = wave_scan(mine, 0, [](int a, int b) { return a + b; });
        for (int e = 0; e < mine; e++) out64[pos + incl - mine + e] = j;
        pos += __builtin_amdgcn_readlane(incl, 63);
      }
    });
    return;
  }
  // The selected columns of a wave are collected in a 128-entry ring in LDS (the histogram is no longer needed: the
  // barrier above lies between its last read and these writes) and leave in full 64-entry, 256-byte stores instead
  // of one partial store per chunk.  LDS operations of one wave complete in order, so the ring needs no barrier.
  int* ring = hist + wave * 128;
  int head = 0, fill = 0;   // wave-uniform
  visit([&](int j, uint32_t key) {
    unsigned long long bk = __builtin_amdgcn_ballot_w64(key > T);
    const unsigned long long beq = __builtin_amdgcn_ballot_w64(key == T);
    if (beq != 0ull && eq_left > 0) {   // keys equal to the threshold: the first eq_left of them by column
      bk |= __builtin_amdgcn_ballot_w64(key == T && lanes_below(beq, lane) < eq_left);
      eq_left = max(0, eq_left - __builtin_popcountll(beq));
    }
    if ((bk >> lane) & 1ull) ring[(head + fill + lanes_below(bk, lane)) & 127] = j;
    fill += __builtin_popcountll(bk);
    if (fill >= 64) {
      out[pos + lane] = ring[(head + lane) & 127];
      head = (head + 64) & 127;
      pos += 64;
      fill -= 64;
    }
  });
  if (lane < fill) out[pos + lane] = ring[(head + lane) & 127];
}

// Keys per thread: every value up to 24 (a row of n keys takes ceil(n / NT) of them: no pass walks more than one
// chunk of padding per wave), then 28 and 32; longer rows are re-read from L2 in every pass.
template <int KPT, int NT, bool UNION>
static bool topk_try(const TopkListParams& p, hipStream_t stream) {
  if (p.n > NT * KPT) return false;
  hipLaunchKernelGGL((topk_token_lists_kernel<KPT, NT, UNION>), dim3(p.rows), dim3(NT), UNION ? (p.n + 1) / 2 * 4 : 0, stream, p);
  return true;
}
template <int NT, bool UNION, int... KPT>
static bool topk_dispatch(const TopkListParams& p, hipStream_t stream, std::integer_sequence<int, KPT...>) {
  return (topk_try<KPT + 1, NT, UNION>(p, stream) || ...);
}

int launch_topk_token_lists(const TopkListParams& p, hipStream_t stream) {
  if (p.rows == 0) return LVAR_OK;
  if (p.more) {
    if (p.n > TOPK_UNION_MAX_N) return LVAR_EUNSUPPORTED;
    topk_dispatch<1024, true>(p, stream, std::make_integer_sequence<int, TOPK_UNION_MAX_N / 1024>{});
    return hipGetLastError() == hipSuccess ? LVAR_OK : LVAR_ELAUNCH;
  }
  // A row is a chain of short phases that end in a barrier.  With at most one row per compute unit half as many keys per
  // thread shorten every phase (1024 against 512 threads, 256 rows: of 6000 keys 8.3 / 11.6 us, of 10521 10.9 / 12.3, of
  // 16384 14.8 / 17.2).  With a second row per compute unit they still win or tie up to 12 keys per thread (512 rows of
  // 10521: 15.7 / 17.0, 257 rows: 14.5 / 14.6), but not beyond: two workgroups then no longer run side by side (512 rows of
  // 12288: 17.9 / 19.8, of 12289: 22.5 / 21.9, of 14336: 25.2 / 22.7; the instances with 13 keys and more are the first
  // with more than 80 scalar registers).  With more rows the 512-thread workgroups of several rows fill each other's
  // gaps better.  (Rows of 512 keys and less have one key per thread either way.)
  const int cus = device_cus();
  const bool few = p.n > 512 && (p.rows <= cus ? p.n <= 16384 : p.rows <= 2 * cus && p.n <= TOPK_SHARED_MAX_N);
  if (few) topk_dispatch<1024, false>(p, stream, std::make_integer_sequence<int, 16>{});
  // 512 threads per row keep a row of up to 16384 keys in registers (KPT keys per thread)
  else if (!topk_dispatch<512, false>(p, stream, std::make_integer_sequence<int, 24>{}) && !topk_try<28, 512, false>(p, stream) && !topk_try<32, 512, false>(p, stream))
    hipLaunchKernelGGL((topk_token_lists_kernel<0, 512, false>), dim3(p.rows), dim3(512), 0, stream, p);
  return hipGetLastError() == hipSuccess ? LVAR_OK : LVAR_ELAUNCH;
}

// ---------------------------------------------------------------------------------------------
// Sparse-step list: out[b,h,g, 0:cnt]       = clamp(src[b,h,gS(g), j / rep], 0, Lk-1)
//                   out[b,h,g, cnt:cnt+L]   = local[g, 0:L]
//                   counts[b,h,g]           = cnt + L
// with gS(g) = clamp(rint((g + 0.5) / Gk * Gs - 0.5), 0, Gs-1) in fp32 (round half to even).
// One workgroup per output row.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void remap_concat_lists_kernel(const RemapListParams p) {
  const int row = blockIdx.x;  // bh * Gk + g
  const int g = row % p.Gk, bh = row / p.Gk;
  const int gs = remap_group(g, p.Gk, p.Gs);
  const int32_t* src = p.src + ((int64_t)bh * p.Gs + gs) * p.src_stride;
  int32_t* out = p.out + (int64_t)row * p.out_stride;
  // A row is a few thousand entries: bound by the round trips to memory, so eight reads go out before the first store (one
  // read per loop turn took 6.1 us for 704 rows of 2700 entries, 5.6 us now).  Clamped reads keep them unconditional.
  constexpr int UN = 8;
  auto copy = [&](int n, int32_t* to, auto&& read) {
    for (int j0 = threadIdx.x; j0 < n; j0 += 256 * UN) {
      int32_t v[UN];
#pragma unroll
      for (int u = 0; u < UN; u++) v[u] = read(min(j0 + u * 256, n - 1));
#pragma unroll
      for (int u = 0; u < UN; u++)
        if (j0 + u * 256 < n) to[j0 + u * 256] = v[u];
    }
  };
  if (p.rep == 1) copy(p.cnt, out, [&](int j) { return max(0, min(p.Lk - 1, src[j])); });
  else copy(p.cnt, out, [&](int j) { return max(0, min(p.Lk - 1, src[j / p.rep])); });
  if (p.local) {
    const int64_t* loc = p.local + (int64_t)g * p.local_stride;
    copy(p.L, out + p.cnt, [&](int j) { return (int32_t)loc[j]; });
  }
  const int total = p.cnt + (p.local ? p.L : 0);
  for (int j = total + threadIdx.x; j < p.zero_to; j += 256) out[j] = 0;   // the rest of the row: defined (zero)
  if (threadIdx.x == 0 && p.counts) p.counts[row] = total;
}

int launch_remap_concat_lists(const RemapListParams& p, hipStream_t stream) {
  if (p.rows == 0) return LVAR_OK;
  hipLaunchKernelGGL(remap_concat_lists_kernel, dim3(p.rows), dim3(256), 0, stream, p);
  return hipGetLastError() == hipSuccess ? LVAR_OK : LVAR_ELAUNCH;
}

// ---------------------------------------------------------------------------------------------
// Mask compaction: ascending columns of the set entries of a uint8 row, count rounded up to a
// multiple with the lowest unset columns as padding.  One 256-thread workgroup per row: every wave
// owns a contiguous quarter of the 64-column chunks, counts its set entries (mask bytes loaded eight
// chunks at a time), learns its output offset from the counts of the waves before it, and writes
// its columns on a second sweep; wave 0 then appends the padding.
// ---------------------------------------------------------------------------------------------
constexpr int MASKLIST_T = 256;

__global__ __launch_bounds__(MASKLIST_T) void mask_to_lists_kernel(const MaskCompactParams p) {
  constexpr int NW = MASKLIST_T / 64, UN = 8;
  __shared__ int wcnt[NW];
  const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint8_t* m = p.mask + (int64_t)row * p.mask_stride;
  int32_t* out = p.indices + (int64_t)row * p.out_stride;
  const int n = p.n;
  const int chunks = (n + 63) >> 6;
  const int cpw = (chunks + NW - 1) / NW;
  const int c_lo = min(chunks, wave * cpw), c_hi = min(chunks, c_lo + cpw);
  // sweep(f): f(first column of the chunk, ballot of the set entries) for every chunk of this wave, ascending
  auto sweep = [&](auto&& f) {
    for (int c0 = c_lo; c0 < c_hi; c0 += UN) {
      uint8_t v[UN];
#pragma unroll
      for (int u = 0; u < UN; u++) {
        const int j = (c0 + u) * 64 + lane;
        v[u] = m[min(j, n - 1)];          // clamped: the load is unconditional, its use is not
      }
#pragma unroll
      for (int u = 0; u < UN; u++) {
        const int j = (c0 + u) * 64 + lane;
        if (c0 + u < c_hi) f((c0 + u) * 64, __builtin_amdgcn_ballot_w64(j < n && v[u] != 0));
      }
    }
  };
  int mine = 0;
  sweep([&](int, unsigned long long bal) { mine += __builtin_popcountll(bal); });
  if (lane == 0) wcnt[wave] = mine;
  __syncthreads();
  int pos = 0, total = 0;
#pragma unroll
  for (int w = 0; w < NW; w++) {
    pos += (w < wave) ? wcnt[w] : 0;
    total += wcnt[w];
  }
  sweep([&](int col0, unsigned long long bal) {
    if ((bal >> lane) & 1ull) out[pos + lanes_below(bal, lane)] = col0 + lane;
    pos += __builtin_popcountll(bal);
  });
  const int mult = max(1, p.multiple_of);
  const int padded = min(n, (total + mult - 1) / mult * mult);
  if (wave == 0) {
    // padding: the lowest unset columns, in ascending order (fewer than `multiple_of` of them)
    int filled = total;
    for (int c = 0; c < chunks && filled < padded; c++) {
      const int j = c * 64 + lane;
      const bool off = j < n && m[j] == 0;
      const unsigned long long bal = __builtin_amdgcn_ballot_w64(off);
      const int at = filled + lanes_below(bal, lane);
      if (off && at < padded) out[at] = j;
      filled = min(padded, filled + __builtin_popcountll(bal));
    }
  }
  if (p.zero_tail)
    for (int t = padded + tid; t < p.out_len; t += MASKLIST_T) out[t] = 0;
  if (tid == 0) p.counts[row] = padded;
}

int launch_mask_to_lists(const MaskCompactParams& p, hipStream_t stream) {
  if (p.rows == 0) return LVAR_OK;
  hipLaunchKernelGGL(mask_to_lists_kernel, dim3(p.rows), dim3(MASKLIST_T), 0, stream, p);
  return hipGetLastError() == hipSuccess ? LVAR_OK : LVAR_ELAUNCH;
}

}  // namespace lvar
