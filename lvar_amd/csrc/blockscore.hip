// Scores of key blocks for gfx950: score[b,h,g,j] = sum over the query rows i of group g and the keys n of block j of
// exp2(q_i.k_n*scale*log2e - lse2_i), from ONE sweep over the logits (row_lse_kernel with SCORES, which see):
//   block_score_finish_kernel   weighs the sums that the sweep kept by exp2(reference - lse2) and adds up the rows of a
//                               group; for callers that rank the blocks it lists the scores too close to the cut for
//                               32-bit sums to tell apart
//   refine_scores_kernel        computes those again the way the column-sum kernel does
// A row with many such scores (keys or queries that repeat, zeros) is handed to the column-sum kernel itself.
#include "common.h"
#include "launch.h"

namespace lvar {

constexpr int SCORE_MAX_GROUP = 1024;   // query rows per group (their weights sit in LDS)
constexpr int REFINE_MAX_ITEMS = 8;     // scores of a row that are computed one by one, see list_close_scores
constexpr int REFINE_MAX_NK = 2048;     // blocks per row that can be ranked (their keys sit in LDS); the limit of the block top-k kernel
// Distance (relative) from which two scores keep their order whichever of the two forms computed them: twice what the forms
// differ by.  The sums and the exponentials: a few units of 2^-24 (4 for N(0, 1) * 0.5 inputs), 16 allowed for the pair.
// The exponents, rounded to 2^-24 of their size: one form rounds (logit - reference) and (reference - statistic), the
// other (logit - statistic).  With D the largest distance of a first reference from the statistic among the rows, N terms
// per score and the score V, the terms' mean distance from their statistics is at most log2(N) - log2(V) (concavity), so
// that the pair differs in the order of 2^-23 (D + log2(N) + |log2(V)|): about 60 units for N(0, 1) * 0.5 inputs, 240 for
// logits of 90 (measured there: 80 for one score, 160 for a pair).
constexpr float REFINE_EPS = 0x1p-20f, REFINE_EPS_EXP = 0x1p-23f;
constexpr float REFINE_FLOOR = 0x1p-120f;   // scores below this are close to one another (terms flush to zero in one form and not in the other)

__device__ __forceinline__ float key_value(uint32_t k) { return __builtin_bit_cast(float, k ^ ((k >> 31) ? 0x80000000u : 0xffffffffu)); }

// One wave per row: appends the row's scores that lie within that distance of the cut of "base blocks plus the best others up
// to `target`" to the work list, when both sides of the cut do.  A score alone costs a wave its operands straight from
// memory, 40 KiB; the column-sum kernel forms all 256 of a row for the price of twenty.  So a row with more than a few is
// listed as a row (the complement of its number) and the column sums of its (batch, head) run: with zero queries (every
// score of every row close) the 24-head 8 x 64 x 64 video lists took 15.3 ms score by score and take 2.6 ms now, against
// 1.6 ms without ties; the launch costs 3 us where no row asks for it.
__device__ __forceinline__ void list_close_scores(const BlockScoreParams& p, const uint32_t* key, const float* wt, int n_wt, int row) {
  const int lane = threadIdx.x & 63, nK = p.nK;
  int others = 0;
  for (int j0 = 0; j0 < nK; j0 += 64) others += __builtin_popcountll(__builtin_amdgcn_ballot_w64(j0 + lane < nK && key[j0 + lane] != 0u));
  const int extra = min(p.target, nK) - (nK - others);
  if (extra <= 0 || extra >= others) return;   // nothing to choose
  auto count = [&](uint32_t v) {
    int n = 0;
    for (int j0 = 0; j0 < nK; j0 += 64) n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(j0 + lane < nK && key[j0 + lane] >= v));
    return n;
  };
  // the extra-th best score: the largest value that at least `extra` keys reach; then the next best
  uint32_t cut = 0u;
  for (int bit = 31; bit >= 0; bit--)
    if (count(cut | (1u << bit)) >= extra) cut |= 1u << bit;
  uint32_t below = 0u;
  if (count(cut) > extra) {
    below = cut;
  } else {
    for (int j = lane; j < nK; j += 64)
      if (key[j] < cut) below = max(below, key[j]);
    for (int d = 32; d > 0; d >>= 1) below = max(below, (uint32_t)__shfl_xor((int)below, d, 64));
  }
  float w = 1.f;   // smallest weight exp2(reference - statistic) of the rows
  for (int t = lane; t < n_wt; t += 64) w = wt[t] > 0.f ? fminf(w, wt[t]) : w;
  for (int d = 32; d > 0; d >>= 1) w = fminf(w, __shfl_xor(w, d, 64));
  const float hi = key_value(cut), lo = key_value(below);
  const float size = __builtin_amdgcn_logf((float)p.group_rows * (float)(p.r.block_stages * 64)) - __builtin_amdgcn_logf(w) + fabsf(__builtin_amdgcn_logf(fmaxf(hi, REFINE_FLOOR)));
  const float eps = fmaf(fmaf(REFINE_EPS_EXP, size, REFINE_EPS), hi, REFINE_FLOOR);
  if (!(hi - lo <= eps)) return;
  auto close = [&](int j) { return j < nK && key[j] != 0u && key_value(key[j]) >= lo - eps && key_value(key[j]) <= hi + eps; };
  int n = 0;
  for (int j0 = 0; j0 < nK; j0 += 64) n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(close(j0 + lane)));
  int* const items = p.r.work + 1 + p.r.B * p.r.H;
  if (n > REFINE_MAX_ITEMS) {
    if (lane == 0) {
      items[atomicAdd(p.r.work, 1)] = ~row;
      atomicAdd(p.r.work + 1 + row / p.G, 1);
    }
    return;
  }
  for (int j = lane; j < nK; j += 64)
    if (close(j)) items[atomicAdd(p.r.work, 1)] = row * nK + j;
}

// Bound by the reads of the kept sums (4 bytes per row and block; B1 H24, 8192 rows x 256 blocks: 58 us, 3.5 TB/s).  One workgroup per
// (batch*head, group) -- per two groups of 32 rows --, 16 lanes x 4 rows per key block, so that every load instruction
// reads 1 KiB in sequence.
template <bool HALF>   // groups of 32 rows: two per 64-row tile of a wave
__global__ __launch_bounds__(256) void block_score_finish_kernel(const BlockScoreParams p) {
  __shared__ __attribute__((aligned(16))) float wt[SCORE_MAX_GROUP];
  extern __shared__ uint32_t keys[];                          // ranking: sort keys of the rows' blocks, 0 for base blocks
  const int tiles = HALF ? 1 : p.group_rows >> 6;             // 64-row tiles of this workgroup
  const int per_bh = HALF ? (p.G + 1) >> 1 : p.G;
  const int bh = blockIdx.x / per_bh, gi = blockIdx.x - bh * per_bh;
  const int row_first = gi * tiles * 64;
  const int have = min(tiles, ((p.r.Lq - row_first) + 63) >> 6);   // those that hold rows
  const int tid = threadIdx.x, lane16 = tid & 15;
  const int64_t row0 = (int64_t)bh * p.r.Lq;
  const int g0 = HALF ? 2 * gi : gi, g = HALF ? g0 + (lane16 >> 3) : g0, nK = p.nK;
  const bool rank = p.target > 0 && nK <= REFINE_MAX_NK;
  for (int t = tid; t < have * 64; t += 256) {
    const int row = row_first + t;
    wt[t] = row < p.r.Lq ? fast_exp2(p.r.first_ref[row0 + row] - p.r.lse2[row0 + row]) : 0.f;
  }
  __syncthreads();
  const bool mine = (lane16 & (HALF ? 7 : 15)) == 0 && g < p.G;
  const float* sums = p.r.tsum + (int64_t)bh * p.r.nrt * 256 * nK + lane16 * 4;   // rows rt64 * 64 ..: at rt64 * nK * 64
  constexpr int U = 4;   // loads in flight per thread
  for (int j0 = tid >> 4; j0 < nK; j0 += 16 * U) {
    float s[U] = {};
    for (int t = 0; t < have; t++) {
      const float* tile = sums + (int64_t)((row_first >> 6) + t) * nK * 64;
      const f32x4 f = *(const f32x4*)(wt + t * 64 + lane16 * 4);
      f32x4 x[U];
#pragma unroll
      for (int u = 0; u < U; u++) x[u] = *(const f32x4*)(tile + min(j0 + 16 * u, nK - 1) * 64);
#pragma unroll
      for (int u = 0; u < U; u++) s[u] += (x[u][0] * f[0] + x[u][1] * f[1]) + (x[u][2] * f[2] + x[u][3] * f[3]);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int j = j0 + 16 * u;
      s[u] = group_sum<HALF ? 8 : 16>(s[u]);
      if (j < nK && mine) {
        p.scores[((int64_t)bh * p.G + g) * nK + j] = s[u];
        if (rank) keys[(g - g0) * nK + j] = (p.base && p.base[(int64_t)g * nK + j]) ? 0u : real_key(s[u]);
      }
    }
  }
  if (!rank) return;
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (wave < (HALF ? 2 : 1) && g0 + wave < p.G) list_close_scores(p, keys + wave * nK, wt + wave * 32, HALF ? 32 : have * 64, bh * p.G + g0 + wave);
}

constexpr int REFINE_WGS = 256;   // of four waves

// One wave per work item.  A score: the value that the block sums of colsum_kernel have (same products, same order of
// additions), so that the selection is the same whichever way the scores were computed.  A row in twenty has such scores at
// 256 blocks, so the operands are read straight from memory.  A row: its scores from those block sums.
template <int D>
__global__ __launch_bounds__(256) void refine_scores_kernel(const BlockScoreParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int KS = D / 16;
  const int lane = threadIdx.x & 63, hh = lane >> 5, r = lane & 31;
  const int nK = p.nK, items = p.r.work[0];
  const f32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int it = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); it < items; it += REFINE_WGS * 4) {
    const int item = __builtin_amdgcn_readfirstlane(p.r.work[1 + p.r.B * p.r.H + it]);
    if (item < 0) {
      const int nkb = (p.r.Lk + 63) >> 6;
      const float* bs = p.r.tsum + (int64_t)~item * nkb;
      for (int j = lane; j < nK; j += 64) {
        const int first = j * p.r.block_stages, end = min(first + p.r.block_stages, nkb);
        float total = bs[first];
        for (int i = first + 1; i < end; i++) total += bs[i];
        p.scores[(int64_t)~item * nK + j] = total;
      }
      continue;
    }
    const int row = item / nK, j = item - row * nK, bh = row / p.G, g = row - bh * p.G, b = bh / p.r.H, h = bh - b * p.r.H;
    const bf16_t* qbase = p.r.q + b * p.r.q_sb + h * p.r.q_sh;
    const bf16_t* kbase = p.r.k + b * p.r.k_sb + (h / p.r.kv_group) * p.r.k_sh;
    const float* lse2 = p.r.lse2 + (int64_t)bh * p.r.Lq;
    float total = 0.f;
    for (int sub = 0; sub < p.r.block_stages; sub++) {
      const int n0 = (j * p.r.block_stages + sub) * 64;
      if (n0 >= p.r.Lk) break;
      bf16x8 kf[2][KS];
#pragma unroll
      for (int nt = 0; nt < 2; nt++) {
        const bf16_t* kp = kbase + (int64_t)min(n0 + nt * 32 + r, p.r.Lk - 1) * p.r.k_sr + hh * 8;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) kf[nt][ks] = *(const bf16x8*)(kp + ks * 16);
      }
      float acc[2] = {0.f, 0.f};
      for (int q0 = g * p.group_rows; q0 < min((g + 1) * p.group_rows, p.r.Lq); q0 += 32) {
        const bf16_t* qp = qbase + (int64_t)min(q0 + r, p.r.Lq - 1) * p.r.q_sr + hh * 8;
        f32x16 s0, s1;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
          const bf16x8 f = *(const bf16x8*)(qp + ks * 16);
          s0 = mfma32(f, kf[0][ks], ks == 0 ? zero : s0);
          s1 = mfma32(f, kf[1][ks], ks == 0 ? zero : s1);
        }
        float pa = 0.f, pb = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const int qrow = q0 + 8 * (i >> 2) + 4 * hh + (i & 3);
          const float ls = lse2[min(qrow, p.r.Lq - 1)];
          const float x0 = fast_exp2(fmaf(s0[i], p.r.c, -ls)), x1 = fast_exp2(fmaf(s1[i], p.r.c, -ls));
          pa += qrow < p.r.Lq ? x0 : 0.f;
          pb += qrow < p.r.Lq ? x1 : 0.f;
        }
        acc[0] += pa;
        acc[1] += pb;
      }
      float val[2];
#pragma unroll
      for (int nt = 0; nt < 2; nt++) {
        const float tot = xhalf_sum(acc[nt]);
        val[nt] = n0 + nt * 32 + r < p.r.Lk ? tot : 0.f;
      }
      const float blk = quad_tree_sum(val[0]) + quad_tree_sum(val[1]);
      total = sub ? total + blk : blk;
    }
    if (lane == 0) p.scores[item] = total;
  }
#endif  // __HIP_DEVICE_COMPILE__
}

int launch_block_scores(const BlockScoreParams& p0, int head_dim, hipStream_t stream) {
  BlockScoreParams p = p0;
  if (p.r.kv_group < 1) p.r.kv_group = 1;
  p.r.nrt = (p.r.Lq + 255) / 256;
  const int st = launch_row_lse(p.r, head_dim, stream);
  if (st != LVAR_OK) return st;
  const int bh = p.r.B * p.r.H;
  const bool rank = p.target > 0 && p.nK <= REFINE_MAX_NK;
  if (p.group_rows == 32)
    hipLaunchKernelGGL(block_score_finish_kernel<true>, dim3(bh * ((p.G + 1) / 2)), dim3(256), rank ? 8 * p.nK : 0, stream, p);
  else
    hipLaunchKernelGGL(block_score_finish_kernel<false>, dim3(bh * p.G), dim3(256), rank ? 4 * p.nK : 0, stream, p);
  if (hipGetLastError() != hipSuccess) return LVAR_ELAUNCH;
  if (rank) {
    ColsumParams c{};
    c.q = p.r.q; c.q_sb = p.r.q_sb; c.q_sh = p.r.q_sh; c.q_sr = p.r.q_sr;
    c.k = p.r.k; c.k_sb = p.r.k_sb; c.k_sh = p.r.k_sh; c.k_sr = p.r.k_sr;
    c.lse2 = p.r.lse2; c.bs = p.r.tsum; c.some = p.r.work + 1;
    c.B = p.r.B; c.H = p.r.H; c.Lq = p.r.Lq; c.Lk = p.r.Lk; c.kv_group = p.r.kv_group;
    c.group_rows = p.group_rows; c.G = p.G; c.c = p.r.c;
    const int st2 = launch_colsum(c, head_dim, stream);
    if (st2 != LVAR_OK) return st2;
    if (head_dim == 128) hipLaunchKernelGGL(refine_scores_kernel<128>, dim3(REFINE_WGS), dim3(256), 0, stream, p);
    else if (head_dim == 64) hipLaunchKernelGGL(refine_scores_kernel<64>, dim3(REFINE_WGS), dim3(256), 0, stream, p);
    else hipLaunchKernelGGL(refine_scores_kernel<256>, dim3(REFINE_WGS), dim3(256), 0, stream, p);
    if (hipGetLastError() != hipSuccess) return LVAR_ELAUNCH;
  }
  return LVAR_OK;
}

}  // namespace lvar
