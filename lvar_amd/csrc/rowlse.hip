// Row statistics for gfx950: lse2[b,h,i] = log2( sum over keys n of exp2(q_i.k_n*scale*log2e) ), the base-2
// log-sum-exp that the column-sum kernel subtracts.
//
// Query-stationary twin of the colsum kernel: a wave keeps 64 query rows (the B operand, Q^T) in registers for its
// whole sweep over the keys; the workgroup (4 waves = 256 rows) streams 64-key K stages through a 2-deep LDS ring
// filled by global->LDS DMA one stage (about 3 us) ahead.  In the 32x32 accumulator a lane owns ONE query row and 16 keys, so
// the sum over keys is an in-register add.
//
// Bound by the vector port (per logit: scale-and-subtract, exp2, add = 19 cycles of one SIMD against 16.6 of its
// matrix pipe), so nothing else may run per logit.  In particular there is no row maximum: the reference that keeps
// exp2 in range is the maximum of the first 64 logits of a row, and once per 64-key stage the running sum is looked
// at and, when it has outgrown LSE_SUM_LIMIT, its exponent moves into the reference (a power of two).  A logit that
// lies more than 2^127 above the running sum overflows the sum; the wave then repeats its rows with a tracked maximum.
// 64 rows per wave instead of the 32 of the attention kernel halve the LDS reads and the L2->LDS fills per flop.
//
// SCORES: the sweep also yields the softmax mass of every key block, summed over groups of query rows.  While a row's
// log-sum-exp is not known yet, the sum of its exponentials over a block of keys can be kept against the row's first
// reference (one float per row and block: 1/128 of the logits at 128-key blocks), and block_score_finish_kernel applies
// exp2(reference - lse2) and adds the rows up.  The second sweep over all logits (the column sums) is not needed then:
// B1 H24 d128, 8192 rows x 32768 keys, 128-key blocks: this sweep 1472 us, finish 58, refinement 14, in place of 1415 for the statistics and 1690 for the column sums.
#include <type_traits>
#include "common.h"
#include "launch.h"

namespace lvar {

constexpr float LSE_SUM_LIMIT = 65536.f;
constexpr int ROW_LSE_STAGES = 2;   // depth of the LDS ring
constexpr float SCORE_REF_LIMIT = 96.f;   // SCORES: largest distance (log2) of a row's reference from its first one
constexpr int ROW_LSE_WGS = 3;      // workgroups per compute unit (head_dim 64 and 128): 168 registers per wave, 32 KiB of LDS

template <int D, bool SCORES>
__global__ __launch_bounds__(256, (D <= 128 ? ROW_LSE_WGS : 1)) void row_lse_kernel(const RowLseParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int KS = D / 16;
  constexpr int ROWB = D * 2, CPR = ROWB / 16;
  constexpr int RPI = 1024 / ROWB, NI = 64 / RPI, SLOTS = NI / 4;
  constexpr int SWD = ROWB >= 256 ? 1 : 256 / ROWB;   // chunk swizzle of row t: (t / SWD) & SWM, 16 rows per period
  constexpr int SWM = ROWB >= 256 ? 15 : CPR - 1;
  constexpr int KTILE = 64 * ROWB;         // one 64-key stage
  constexpr int NSTAGE = ROW_LSE_STAGES, PF = NSTAGE - 1;   // PF stages in flight ahead of the one being used
  extern __shared__ __attribute__((aligned(1024))) char smem[];  // NSTAGE * KTILE bytes

  // consecutive workgroup ids are dealt round-robin to the 8 XCDs: each XCD walks a contiguous range
  const int per_xcd = gridDim.x >> 3;
  const int w = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (SCORES && blockIdx.x == 0)
    for (int i = threadIdx.x; i <= p.B * p.H; i += 256) p.work[i] = 0;
  if (w >= p.total_wg) return;
  // workgroup = (batch*head, key range, tile of 256 query rows)
  const int per_bh = p.nrt * p.splits;
  // (the quotients are formed on the vector ALU: moved to scalar registers, so are the addresses that hang on them)
  const int bh = __builtin_amdgcn_readfirstlane(w / per_bh), rem = w - bh * per_bh;
  const int sp = __builtin_amdgcn_readfirstlane(rem / p.nrt), rt = rem - sp * p.nrt;
  const int b = __builtin_amdgcn_readfirstlane(bh / p.H), h = bh - b * p.H;
  const int koff = __builtin_amdgcn_readfirstlane(sp * p.split_keys);       // first key of this range (a multiple of 64)
  const int Lk_l = min(p.Lk, koff + p.split_keys) - koff;                   // keys of this range
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = lane >> 5, r = lane & 31;
  const int n0 = rt * 256 + wave * 64;     // first query row of this wave
  const float c = p.c;

  const bf16_t* kbase = p.k + b * p.k_sb + __builtin_amdgcn_readfirstlane(h / p.kv_group) * p.k_sh;   // grouped-query attention: shared key heads
  // buffer descriptor that ends with the last key row: the rows of a ragged last stage beyond it read as zeros
  const int k_srb = (int)p.k_sr * 2;
  const uint64_t ka = (uint64_t)kbase;
  const i32x4 krsrc = {__builtin_amdgcn_readfirstlane((int)(uint32_t)ka), __builtin_amdgcn_readfirstlane((int)(uint32_t)((ka >> 32) & 0xffffu)),
                       __builtin_amdgcn_readfirstlane((p.Lk - 1) * k_srb + ROWB), 0x00020000};
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LVAR_LDS char*)smem;
  const int lrow = lane / CPR, lcs = lane % CPR;

  // lane offset of a fill: row within the first instruction(s) of this wave, swizzled chunk; slots a whole swizzle
  // period (16 rows) apart share it, tile and slot move the scalar offset
  constexpr int PER = (4 * RPI >= 16) ? 1 : 16 / (4 * RPI);
  static_assert((PER * 4 * RPI) % 16 == 0 && SLOTS % PER == 0, "slots PER apart must be whole swizzle periods apart");
  int fill_voff[PER];
#pragma unroll
  for (int ph = 0; ph < PER; ph++) {
    const int trow = (wave + 4 * ph) * RPI + lrow;
    fill_voff[ph] = trow * k_srb + ((lcs ^ ((trow / SWD) & SWM)) << 4);
  }
  auto issue_stage = [&](int s) {
    const uint32_t dst = lds0 + (s & (NSTAGE - 1)) * KTILE;
#pragma unroll
    for (int sl = 0; sl < SLOTS; sl++) {
      const int soff = (koff + s * 64 + (sl / PER) * PER * 4 * RPI) * k_srb;
      const uint32_t m0v = dst + (wave + sl * 4) * 1024;
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" : : "s"(m0v), "v"(fill_voff[sl % PER]), "s"(krsrc), "s"(soff) : "memory");
    }
  };
  // (the ring has two stages, so nothing younger than the stage that is waited for is in flight)
  static_assert(PF == 1, "one stage ahead");
  auto wait_fills = [&] { __builtin_amdgcn_s_waitcnt(0x0f70); };   // vmcnt(0)

  const int S = (Lk_l + 63) >> 6;          // stages of this range
  // the ring filled; with the query fragments one round trip to memory
#pragma unroll
  for (int s = 0; s < NSTAGE; s++)
    if (s < S) issue_stage(s);
  if (n0 >= p.Lq) {
    // A wave without rows (the last row tile of a slice) keeps its part of the fills and meets
    // the barriers (1600 rows: 25 of 28 waves have rows; with the column sums behind it 124.7 -> 123.1 us).
    wait_fills();
    __syncthreads();
    if (S > 1) __syncthreads();
    for (int s = 1; s + 1 < S; s++) {
      if (s + PF < S) issue_stage(s + PF);
      wait_fills();
      __syncthreads();
    }
    return;
  }

  // stationary Q^T fragments: lane holds query row n0 + nt*32 + r, d = ks*16 + 8*hh .. +7
  const bf16_t* qbase = p.q + b * p.q_sb + h * p.q_sh;
  bf16x8 qf[2][KS];
#pragma unroll
  for (int nt = 0; nt < 2; nt++) {
    const int qrow = min(n0 + nt * 32 + r, p.Lq - 1);
    const bf16_t* qp = qbase + (int64_t)qrow * p.q_sr + hh * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) qf[nt][ks] = *(const bf16x8*)(qp + ks * 16);
  }

  const int U = (Lk_l + 31) >> 5;          // 32-key tiles
  const int kbase_l = r * ROWB + ((hh ^ ((r / SWD) & SWM)) << 4);
  // Reference and sum of this lane's half of the keys, per query row.  The sum runs in the order of the attention
  // kernel's row sum (even and odd elements of a 64-key stage apart; the two halves of the last stage apart), with the
  // same first reference: while neither kernel moves its reference (the attention kernel does for a logit 2^8 above it,
  // this one for a sum above LSE_SUM_LIMIT), statistics of one key range have the bits that the attention kernel gives.
  float m[2], l[2] = {0.f, 0.f}, la[2], lb[2];
  // SCORES: stages left in the open key block, and its sum against the first reference; lane = row of the wave (both
  // halves of the keys added up), one register.  (Two sums, one per half, spill; sums in LDS cost the loop 40 %: an
  // LDS atomic takes about 100 cycles.)  The first references sit in LDS and are read once a reference has moved.
  int left = p.block_stages, blk = 0;
  float bsum = 0.f;
  bool moved = false;
  float* const tp = SCORES ? p.tsum + ((int64_t)w * 4 + wave) * p.key_blocks * 64 : nullptr;
  auto lane_id = []() {   // formed where it is needed: every register counts in the loop
    int ln;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
    return ln;
  };
  auto first = [&](int nt) -> LVAR_LDS float& { return ((LVAR_LDS float*)(smem + NSTAGE * KTILE))[wave * 128 + nt * 64 + lane_id()]; };
  auto add_block = [&](float t0, float t1) {
    if (moved) {
      t0 *= fast_exp2(m[0] - first(0));
      t1 *= fast_exp2(m[1] - first(1));
    }
    const auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, t0), __builtin_bit_cast(int, t1), false, false);
    bsum += __builtin_bit_cast(float, (int)sw[0]) + __builtin_bit_cast(float, (int)sw[1]);
  };
  auto emit = [&]() {
    tp[blk * 64 + lane_id()] = bsum;
    bsum = 0.f;
    blk++;
    left = p.block_stages;
  };
  // after a stage: when a sum has outgrown the limit its exponent moves into the reference
  auto renorm = [&]() {
    if (__builtin_amdgcn_ballot_w64(fmaxf(l[0], l[1]) > LSE_SUM_LIMIT) != 0) {
#pragma unroll
      for (int nt = 0; nt < 2; nt++) {
        // exponent of the sum (an infinite one stays infinite whatever is taken off)
        const int e = (int)((__builtin_bit_cast(uint32_t, l[nt]) >> 23) & 255u) - 127;
        const int d = (l[nt] > LSE_SUM_LIMIT && e < 128) ? e : 0;
        // (the reference rounds when the exponent is added to it: what it has not moved stays with the sums)
        const float mn = m[nt] + (float)d, rest = fast_exp2((float)d - (mn - m[nt]));
        l[nt] = __builtin_amdgcn_ldexpf(l[nt], -d) * rest;
        m[nt] = mn;
      }
      moved = true;
    }
  };
  const f32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};   // constant addend of the first MFMA
  // accumulator i of this lane is tile key 8*(i/4) + 4*hh + (i%4): keys at or beyond the limit take no part
  auto mask_tile = [&](int u, f32x16& s0, f32x16& s1) {
    const int lim = Lk_l - u * 32 - 4 * hh;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const bool ok = (8 * (i >> 2) + (i & 3)) < lim;
      s0[i] = ok ? s0[i] : -INFINITY;
      s1[i] = ok ? s1[i] : -INFINITY;
    }
  };
  auto tile_max = [&](const f32x16& s) -> float {
    float a = s[0], bmx = s[1];
#pragma unroll
    for (int i = 2; i < 16; i += 2) { a = fmaxf(a, s[i]); bmx = fmaxf(bmx, s[i + 1]); }
    return fmaxf(a, bmx);
  };

  // S(u) = K_tile(u) Q^T -> (n0a, n1a) on the matrix cores, nothing beside it
  auto qk_tile = [&](int u, f32x16& n0a, f32x16& n1a) {
    const char* kb = smem + ((u >> 1) & (NSTAGE - 1)) * KTILE + (u & 1) * 32 * ROWB;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      const bf16x8 f = *(const bf16x8*)(kb + (kbase_l ^ (ks << 5)));
      n0a = mfma32(f, qf[0][ks], ks == 0 ? zero : n0a);
      n1a = mfma32(f, qf[1][ks], ks == 0 ? zero : n1a);
    }
  };
  // exponentials of a tile of the last stage, or of one without a successor: one sum
  auto tile_sum = [&](const f32x16& s0, const f32x16& s1, float (&to)[2]) {
    to[0] = to[1] = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      to[0] += fast_exp2(fmaf(s0[i], c, -m[0]));
      to[1] += fast_exp2(fmaf(s1[i], c, -m[1]));
    }
  };

  // S(u) on the matrix cores, the exponentials of tile u-1 from (c0, c1) on the vector ALU as a three-stage pipeline
  // over the MFMA steps (scale | exp2 | add), interleaved by hand.  One per 64-key stage opens the two sums (tile u-1
  // is the first of its stage), the other closes them; `whole`: the first tile of the last stage, one sum.
  // (`buf`: the stage's place in the ring, a constant in the loop of SCORES)
  auto step = [&](auto buf, int u, f32x16& n0a, f32x16& n1a, const f32x16& c0, const f32x16& c1, auto opens, auto whole) {
    constexpr bool OPENS = decltype(opens)::value, WHOLE = decltype(whole)::value;
    const char* kb = smem + buf * KTILE + (u & 1) * 32 * ROWB;
    constexpr int AHEAD = 2;
    bf16x8 frag[KS];
#pragma unroll
    for (int j = 0; j < AHEAD && j < KS; j++) frag[j] = *(const bf16x8*)(kb + (kbase_l ^ (j << 5)));
    constexpr int EPS = 16 / KS;
    const float negm0 = -m[0], negm1 = -m[1];
    if (OPENS) la[0] = la[1] = lb[0] = lb[1] = 0.f;
    float xs0[16], xs1[16];
    auto st_scale = [&](int g) {
#pragma unroll
      for (int e = 0; e < EPS; e++) {
        const int i = g * EPS + e;
        xs0[i] = fmaf(c0[i], c, negm0);
        xs1[i] = fmaf(c1[i], c, negm1);
      }
    };
    auto st_exp = [&](int g) {
#pragma unroll
      for (int e = 0; e < EPS; e++) {
        const int i = g * EPS + e;
        xs0[i] = fast_exp2(xs0[i]);
        xs1[i] = fast_exp2(xs1[i]);
      }
    };
    auto st_add = [&](int g) {
#pragma unroll
      for (int e = 0; e < EPS; e++) {
        const int i = g * EPS + e;
        if (WHOLE || (i & 1) == 0) { la[0] += xs0[i]; la[1] += xs1[i]; }
        else { lb[0] += xs0[i]; lb[1] += xs1[i]; }
      }
    };
    st_scale(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      if (ks + AHEAD < KS) frag[ks + AHEAD] = *(const bf16x8*)(kb + (kbase_l ^ ((ks + AHEAD) << 5)));
      n0a = mfma32(frag[ks], qf[0][ks], ks == 0 ? zero : n0a);
      n1a = mfma32(frag[ks], qf[1][ks], ks == 0 ? zero : n1a);
      if (ks >= 1) st_add(ks - 1);
      st_exp(ks);
      if (ks + 1 < KS) st_scale(ks + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    st_add(KS - 1);
    // (the sums are wanted here: left to itself the compiler moves exponentials into the next step, behind its MFMAs)
    if (SCORES && OPENS) asm volatile("" : "+v"(la[0]), "+v"(la[1]), "+v"(lb[0]), "+v"(lb[1]));
    if (!OPENS) {
      const float t0 = la[0] + lb[0], t1 = la[1] + lb[1];
      l[0] += t0;
      l[1] += t1;
      if (SCORES) add_block(t0, t1);
      renorm();
    }
  };
  using yes = std::true_type;
  using no = std::false_type;

  // prologue: the first stage gives the reference
  wait_fills();
  __syncthreads();
  f32x16 sa0, sa1, sb0, sb1;
  qk_tile(0, sa0, sa1);
  qk_tile(1, sb0, sb1);
  if (S == 1) { mask_tile(0, sa0, sa1); mask_tile(1, sb0, sb1); }
  m[0] = xhalf_max(fmaxf(tile_max(sa0), tile_max(sb0))) * c;
  m[1] = xhalf_max(fmaxf(tile_max(sa1), tile_max(sb1))) * c;
  if (SCORES) {
    first(0) = m[0];
    first(1) = m[1];
  }
  if (S > 1) {
    la[0] = la[1] = lb[0] = lb[1] = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const float x0 = fast_exp2(fmaf(sa0[i], c, -m[0])), x1 = fast_exp2(fmaf(sa1[i], c, -m[1]));
      if (i & 1) { lb[0] += x0; lb[1] += x1; } else { la[0] += x0; la[1] += x1; }
    }
    __syncthreads();   // every wave has read stage 0: its place may be filled
    auto stage = [&](auto buf, int s) {
      // (before the fills, so that one wait covers both, and with nothing conditional behind a step: the compiler
      // moves a step's exponentials past it, out of the shadow of its matrix instructions)
      if (SCORES && left == 0) emit();
      if (s + PF < S) issue_stage(s + PF);
      step(buf, 2 * s, sa0, sa1, sb0, sb1, no{}, no{});
      if (SCORES) left--;
      step(buf, 2 * s + 1, sb0, sb1, sa0, sa1, yes{}, no{});
      wait_fills();
      __syncthreads();
    };
    if constexpr (SCORES) {
      // two stages per turn: the place in the ring is part of the reads, which saves eight vector additions per stage
      // (B1 H24 d128, 8 x 64 x 64 tokens, lists in all: 1526 -> 1515 us; H8, 4 x 48 x 48: 183.9 -> 180.6; H16 d64, 4 x 64 x 64: 254 -> 249).  Without SCORES
      // the registers that this takes spill around the loop, and short sweeps lose as much (1600 x 4121: +1 us).
      using P0 = std::integral_constant<int, 0>;
      using P1 = std::integral_constant<int, 1>;
      int s = 1;
      for (; s + 2 < S; s += 2) {
        stage(P1{}, s);
        stage(P0{}, s + 1);
      }
      if (s + 1 < S) stage(P1{}, s);
    } else {
      for (int s = 1; s + 1 < S; s++) stage(s & (NSTAGE - 1), s);
    }
    const int buf = (S - 1) & (NSTAGE - 1);
    if (SCORES && left == 0) emit();
    step(buf, 2 * S - 2, sa0, sa1, sb0, sb1, no{}, no{});
    if (SCORES && --left == 0) emit();
    if (U & 1) {
      mask_tile(U - 1, sa0, sa1);
      tile_sum(sa0, sa1, la);
      lb[0] = lb[1] = 0.f;
    } else {
      step(buf, 2 * S - 1, sb0, sb1, sa0, sa1, yes{}, yes{});
      mask_tile(U - 1, sb0, sb1);
      tile_sum(sb0, sb1, lb);
    }
  } else {
    tile_sum(sa0, sa1, la);
    tile_sum(sb0, sb1, lb);
  }
  l[0] += la[0] + lb[0];
  l[1] += la[1] + lb[1];
  if (SCORES) {
    add_block(la[0] + lb[0], la[1] + lb[1]);
    emit();
  }
  // The last stage too: a sum of up to 2^127 against a reference that lies as far below the other half of the row, or
  // below another key range, would vanish from the weighted sum of the two; and SCORES judges the distance of the
  // statistic, not of the reference before the last keys, from the first reference.
  renorm();

  const bool overflow = __builtin_amdgcn_ballot_w64(!(fmaxf(l[0], l[1]) < INFINITY)) != 0;
  bool again = overflow;
  if (SCORES) again = again || __builtin_amdgcn_ballot_w64(fmaxf(m[0] - first(0), m[1] - first(1)) > SCORE_REF_LIMIT) != 0;
  const float m_sweep[2] = {m[0], m[1]}, l_sweep[2] = {l[0], l[1]};
  if (again) {
    // a sum has overflowed: this wave's rows again, straight from memory, with the maximum tracked tile by tile
    auto tile_mem = [&](int u) {
      const bf16_t* kp = kbase + (int64_t)min(koff + u * 32 + r, p.Lk - 1) * p.k_sr + hh * 8;
      sa0 = zero;
      sa1 = zero;
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        const bf16x8 kfr = *(const bf16x8*)(kp + ks * 16);
        sa0 = mfma32(kfr, qf[0][ks], sa0);
        sa1 = mfma32(kfr, qf[1][ks], sa1);
      }
      mask_tile(u, sa0, sa1);
    };
    l[0] = l[1] = 0.f;
    m[0] = m[1] = -1.0e30f;
    for (int u = 0; u < U; u++) {
      tile_mem(u);
#pragma unroll
      for (int nt = 0; nt < 2; nt++) {
        const f32x16& s = nt ? sa1 : sa0;
        const float m_new = fmaxf(m[nt], tile_max(s) * c);
        float t = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i++) t += fast_exp2(fmaf(s[i], c, -m_new));
        l[nt] = fmaf(l[nt], fast_exp2(m[nt] - m_new), t);
        m[nt] = m_new;
      }
    }
    if (SCORES) {
      // and the block sums against that maximum (`blk` is past the end: the stores of the first sweep are overwritten)
#pragma unroll
      for (int nt = 0; nt < 2; nt++) {
        const float mm = xhalf_max(m[nt]);
        l[nt] *= fast_exp2(m[nt] - mm);
        m[nt] = first(nt) = mm;
      }
      blk = 0;
      moved = false;
      for (int u = 0; u < U; u++) {
        tile_mem(u);
        float t0 = 0.f, t1 = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
          t0 += fast_exp2(fmaf(sa0[i], c, -m[0]));
          t1 += fast_exp2(fmaf(sa1[i], c, -m[1]));
        }
        add_block(t0, t1);
        if (u + 1 == U || (u + 1) % (2 * p.block_stages) == 0) emit();
      }
      // the statistic of a sweep that was only repeated for its block sums stands: it has the bits of the one without SCORES
      if (!overflow) {
#pragma unroll
        for (int nt = 0; nt < 2; nt++) {
          m[nt] = m_sweep[nt];
          l[nt] = l_sweep[nt];
        }
      }
    }
  }

  // the two lanes of a row add up; one range: the statistic itself, several: reference and sum of this range
  const int64_t row0 = ((int64_t)b * p.H + h) * p.Lq;
  const int64_t rows_all = (int64_t)p.B * p.H * p.Lq;
#pragma unroll
  for (int nt = 0; nt < 2; nt++) {
    const float mm = xhalf_max(l[nt] > 0.f ? m[nt] : -1.0e30f);
    const float ll = xhalf_sum(l[nt] * fast_exp2(fminf(m[nt] - mm, 0.f)));
    const int row = n0 + nt * 32 + r;
    if (hh == 0 && row < p.Lq) {
      if (SCORES) p.first_ref[row0 + row] = first(nt);
      if (p.splits == 1) {
        p.lse2[row0 + row] = mm + __builtin_amdgcn_logf(ll);
      } else {
        p.part[(int64_t)(2 * sp) * rows_all + row0 + row] = mm;
        p.part[(int64_t)(2 * sp + 1) * rows_all + row0 + row] = ll;
      }
    }
  }
#endif  // __HIP_DEVICE_COMPILE__
}

// lse2 of a row from the references and sums of its key ranges
__global__ __launch_bounds__(256) void row_lse_merge_kernel(const float* part, float* lse2, int64_t rows, int splits) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= rows) return;
  float m[ROW_LSE_MAX_SPLITS], l[ROW_LSE_MAX_SPLITS];
#pragma unroll
  for (int s = 0; s < ROW_LSE_MAX_SPLITS; s++) {
    m[s] = s < splits ? part[(int64_t)(2 * s) * rows + i] : -INFINITY;
    l[s] = s < splits ? part[(int64_t)(2 * s + 1) * rows + i] : 0.f;
  }
  float mm = m[0];
#pragma unroll
  for (int s = 1; s < ROW_LSE_MAX_SPLITS; s++) mm = fmaxf(mm, m[s]);
  float ll = 0.f;
#pragma unroll
  for (int s = 0; s < ROW_LSE_MAX_SPLITS; s++) ll = fmaf(l[s], fast_exp2(m[s] - mm), ll);
  lse2[i] = mm + __builtin_amdgcn_logf(ll);
}

// lse2 = M + log2(L) from the statistics of a dense pass
__global__ __launch_bounds__(256) void lse2_from_stats_kernel(const float* M, const float* L, float* lse2, int64_t rows) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < rows) lse2[i] = M[i] + __builtin_amdgcn_logf(L[i]);
}

int launch_lse2_from_stats(const float* M, const float* L, float* lse2, int64_t rows, hipStream_t stream) {
  hipLaunchKernelGGL(lse2_from_stats_kernel, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, stream, M, L, lse2, rows);
  return hipGetLastError() == hipSuccess ? LVAR_OK : LVAR_ELAUNCH;
}

// Key ranges per row tile: workgroups are handed to the resident slots as slots fall free, so a
// launch takes its total work over the slots plus a part of the longest workgroup while the chip drains (the model of
// the colsum launch, in 64-key stages of about 3 us), and the merge of several ranges costs a launch of its own.
int row_lse_splits(int B, int H, int Lq, int Lk) {
  const int base_wg = B * H * ((Lq + 255) / 256), slots = ROW_LSE_WGS * device_cus(), stages = (Lk + 63) / 64;
  if (slots <= 0 || base_wg >= 4 * slots) return 1;
  int best_n = 1;
  double best = -1.0;
  for (int s = 1; s <= ROW_LSE_MAX_SPLITS && s <= stages; s++) {
    const int per = (stages + s - 1) / s;
    if (s > 1 && per < 4) break;
    const int n = (stages + per - 1) / per;
    const double work = (double)base_wg * (stages + 1.5 * n) / slots;
    const double cost = (work > per + 1.5 ? work : per + 1.5) + 0.4 * (per + 1.5) + (n > 1 ? 1.5 : 0.0);
    if (best < 0.0 || cost < best) { best = cost; best_n = n; }
  }
  return best_n;
}

template <int D, bool SCORES>
static int launch_rl(const RowLseParams& p0, hipStream_t stream) {
  RowLseParams p = p0;
  if (p.kv_group < 1) p.kv_group = 1;
  p.nrt = (p.Lq + 255) / 256;
  const int stages = (p.Lk + 63) / 64;
  p.splits = p.part ? row_lse_splits(p.B, p.H, p.Lq, p.Lk) : 1;
  const int per = (stages + p.splits - 1) / p.splits;
  p.splits = (stages + per - 1) / per;                 // ranges that hold keys
  p.split_keys = per * 64;
  p.total_wg = p.B * p.H * p.nrt * p.splits;
  const int grid = ((p.total_wg + 7) / 8) * 8;
  constexpr int SMEM = ROW_LSE_STAGES * 64 * D * 2 + (SCORES ? 4 * 128 * 4 : 0);
  static std::atomic<uint64_t> lds_ready{0};
  if (!ensure_lds_limit((const void*)row_lse_kernel<D, SCORES>, SMEM, lds_ready)) return LVAR_ELAUNCH;
  hipLaunchKernelGGL((row_lse_kernel<D, SCORES>), dim3(grid), dim3(256), SMEM, stream, p);
  if (hipGetLastError() != hipSuccess) return LVAR_ELAUNCH;
  if (p.splits > 1) {
    const int64_t rows = (int64_t)p.B * p.H * p.Lq;
    hipLaunchKernelGGL(row_lse_merge_kernel, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, stream, p.part, p.lse2, rows, p.splits);
    if (hipGetLastError() != hipSuccess) return LVAR_ELAUNCH;
  }
  return LVAR_OK;
}

int launch_row_lse(const RowLseParams& p, int head_dim, hipStream_t s) {
  if (p.tsum) {
    if (head_dim == 128) return launch_rl<128, true>(p, s);
    if (head_dim == 64) return launch_rl<64, true>(p, s);
    if (head_dim == 256) return launch_rl<256, true>(p, s);
    return LVAR_EUNSUPPORTED;
  }
  if (head_dim == 128) return launch_rl<128, false>(p, s);
  if (head_dim == 64) return launch_rl<64, false>(p, s);
  if (head_dim == 256) return launch_rl<256, false>(p, s);
  return LVAR_EUNSUPPORTED;
}

}  // namespace lvar
