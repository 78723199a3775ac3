// Colsum kernel for gfx950: cs[b,h,g,n] = sum over the query rows i of group g of
// exp2(q_i.k_n*scale*log2e - lse2_i), with lse2 = M + log2(L) the base-2 log-sum-exp of row i.
//
// Key-stationary decomposition: a wave keeps one 64-key block (the B operand, K^T) in registers
// for the whole sweep over Lq; the workgroup (4 waves = 256 keys) streams 64-row Q stages and their
// lse2 through a 2-deep LDS ring filled by global->LDS DMA one stage ahead.  In the 32x32
// accumulator a lane owns ONE key column and 16 query rows, so the reduction over queries is an
// in-register add, one exchange with lane^32 at each group boundary and a single plain store per
// (group, key): no atomics, no partial buffers, and a summation order fixed by the shapes alone.
// The per-64-key block sums fall out of the same registers (one wave = one key block).
//
// Inner loop, software-pipelined by hand: while the matrix cores compute S(u) = Q_tile(u) K^T for
// 32-row tile u (16 MFMA for d = 128), the vector ALU turns S(u-1) into probabilities and adds them
// to the column accumulators.
#include <type_traits>
#include "common.h"
#include "launch.h"

namespace lvar {

constexpr int CS_WGS = 3;   // workgroups per compute unit (head_dim 64 and 128): 168 registers per wave, 33 KiB of LDS

template <int D, bool SOME>
__global__ __launch_bounds__(256, (D <= 128 ? CS_WGS : 1)) void colsum_kernel(const ColsumParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int KS = D / 16;
  constexpr int ROWB = D * 2, CPR = ROWB / 16;
  constexpr int RPI = 1024 / ROWB, NI = 64 / RPI, SLOTS = NI / 4;
  constexpr int SWD = ROWB >= 256 ? 1 : 256 / ROWB;   // chunk swizzle of row t: (t / SWD) & SWM, 16 rows per period
  constexpr int SWM = ROWB >= 256 ? 15 : CPR - 1;
  constexpr int QTILE = 64 * ROWB;         // one 64-row Q stage
  constexpr int NSTAGE = 2, NLSE = 4;      // ring depths
  constexpr int LSE_OFF = NSTAGE * QTILE;  // lse2 ring: NLSE x 64 floats
  extern __shared__ __attribute__((aligned(1024))) char smem[];  // NSTAGE * QTILE + NLSE * 256 bytes

  const int per_xcd = gridDim.x >> 3;
  const int w = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (w >= p.total_wg) return;
  // workgroup = (batch*head, key tile of 256 keys, range of query groups): the query axis is cut at group
  // boundaries when the plain grid would fill the chip unevenly; every range writes its own groups of cs
  const int per_bh = p.nkt * p.q_splits;
  // (the quotients are formed on the vector ALU: moved to scalar registers, so are the addresses that hang on them)
  const int bh = __builtin_amdgcn_readfirstlane(w / per_bh), rem = w - bh * per_bh;
  const int kt = __builtin_amdgcn_readfirstlane(rem / p.q_splits), sp = rem - kt * p.q_splits;
  if (SOME && p.some[bh] == 0) return;
  const int b = __builtin_amdgcn_readfirstlane(bh / p.H), h = bh - b * p.H;
  const int qoff = __builtin_amdgcn_readfirstlane(sp * p.split_rows);   // first query row of this range (a multiple of 64 and of group_rows)
  const int Lq_l = min(p.Lq, qoff + p.split_rows) - qoff;   // rows of this range
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = lane >> 5, r = lane & 31;
  const int kblk = kt * 4 + wave;  // 64-key block owned by this wave
  const int n0 = kblk * 64;
  const float c = p.c;
  // the lane number, formed where it is needed: every register counts in the loop
  auto lane_id = []() {
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
  };

  // stationary K^T fragments: lane holds key column n0 + nt*32 + r, d = ks*16 + 8*hh .. +7
  const bf16_t* kbase = p.k + b * p.k_sb + __builtin_amdgcn_readfirstlane(h / p.kv_group) * p.k_sh;   // grouped-query attention: shared key heads
  bf16x8 kf[2][KS];
#pragma unroll
  for (int nt = 0; nt < 2; nt++) {
    const int krow = min(n0 + nt * 32 + r, p.Lk - 1);
    const bf16_t* kp = kbase + (int64_t)krow * p.k_sr + hh * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) kf[nt][ks] = *(const bf16x8*)(kp + ks * 16);
  }

  // buffer descriptors that end with the last row: what a ragged last stage fetches beyond it reads as zeros (the rows
  // are masked); stores beyond the last key of a row of cs are dropped
  auto make_rsrc = [](const void* base, int bytes) -> i32x4 {
    const uint64_t a = (uint64_t)base;
    i32x4 rs = {__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
                __builtin_amdgcn_readfirstlane((int)(uint32_t)((a >> 32) & 0xffffu)), __builtin_amdgcn_readfirstlane(bytes), 0x00020000};
    return rs;
  };
  const i32x4 qrsrc = make_rsrc(p.q + b * p.q_sb + h * p.q_sh, (p.Lq - 1) * (int)p.q_sr * 2 + ROWB);
  const i32x4 lrsrc = make_rsrc(p.lse2 + ((int64_t)b * p.H + h) * p.Lq, p.Lq * 4);
  const int q_srb = (int)p.q_sr * 2;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LVAR_LDS char*)smem;
  const int lrow = lane / CPR, lcs = lane % CPR;

  // global->LDS fill of stage s (Q rows s*64 .. +63, chunk-swizzled; lse2 by wave 0)
  // lane offset of a Q fill: row within the first instruction(s) of this wave, swizzled chunk.  The swizzle
  // repeats every 16 rows and instruction i = wave + 4 * slot covers rows i * RPI ..: slots a whole period apart
  // share the lane offset (PER = 1: all of them; head_dim 256 has two rows per instruction and PER = 2).
  constexpr int PER = (4 * RPI >= 16) ? 1 : 16 / (4 * RPI);
  static_assert((PER * 4 * RPI) % 16 == 0 && SLOTS % PER == 0, "slots PER apart must be whole swizzle periods apart");
  int fill_voff[PER];
#pragma unroll
  for (int ph = 0; ph < PER; ph++) {
    const int trow = (wave + 4 * ph) * RPI + lrow;
    fill_voff[ph] = trow * q_srb + ((lcs ^ ((trow / SWD) & SWM)) << 4);
  }
  auto issue_stage = [&](int s) {
    const uint32_t dst = lds0 + (s & (NSTAGE - 1)) * QTILE;
#pragma unroll
    for (int sl = 0; sl < SLOTS; sl++) {
      const int soff = (qoff + s * 64 + (sl / PER) * PER * 4 * RPI) * q_srb;
      const uint32_t m0v = dst + (wave + sl * 4) * 1024;
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" : : "s"(m0v), "v"(fill_voff[sl % PER]), "s"(qrsrc), "s"(soff) : "memory");
    }
    if (wave == 0) {
      const uint32_t m0v = lds0 + LSE_OFF + (s & (NLSE - 1)) * 256;
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds" : : "s"(m0v), "v"(lane_id() * 4), "s"(lrsrc), "s"((qoff + s * 64) * 4) : "memory");
    }
  };
  constexpr auto vm = [](int n) constexpr { return 0x0f70 | (n & 15) | (((n >> 4) & 3) << 14); };   // expcnt, lgkmcnt: don't wait
  // wait for this wave's fills; `stores` memory operations issued after them may still be in flight
  auto wait_fills = [&](int stores) {
    __builtin_amdgcn_sched_barrier(0);
    if (stores >= 3) __builtin_amdgcn_s_waitcnt(vm(3));
    else if (stores == 2) __builtin_amdgcn_s_waitcnt(vm(2));
    else if (stores == 1) __builtin_amdgcn_s_waitcnt(vm(1));
    else __builtin_amdgcn_s_waitcnt(vm(0));
  };

  const int S = (Lq_l + 63) >> 6;          // stages of this range
  const int U = (Lq_l + 31) >> 5;          // 32-row tiles
  // both stages of the ring and the key fragments are one round trip to memory
  issue_stage(0);
  if (S > 1) issue_stage(1);
  if (n0 >= p.Lk) {
    // A wave without keys (the last key tile of a slice; three of its four waves at 4121, 6425 and 10521 keys) keeps its part
    // of the fills and meets the barriers.  With the first two stages requested together, B2 H16 d128: 1600 x 4121 68.2 ->
    // 67.3 us, 2304 x 6425 126.4 -> 125.0, 4096 x 10521 347.6 -> 345.0.  (Starting these tiles last is 0.3 % slower.)
    wait_fills(0);
    __syncthreads();
    for (int s = 0; s < S; s++) {
      if (s > 0 && s + 1 < S) issue_stage(s + 1);
      wait_fills(0);
      __syncthreads();
    }
    return;
  }

  float* csp = p.cs ? p.cs + ((int64_t)b * p.H + h) * p.G * (int64_t)p.Lk : nullptr;
  float* bsp = p.bs ? p.bs + ((int64_t)b * p.H + h) * p.G * (int64_t)p.nkb : nullptr;
  int flush_stores = 0;   // stores of the flushes since the last fill
  // store the finished column sums of group g and reset the accumulators
  auto flush = [&](int g, float (&acc)[2]) {
    const int ln = lane_id(), hh = ln >> 5, r = ln & 31;
    float blk = 0.f, val[2];
#pragma unroll
    for (int nt = 0; nt < 2; nt++) {
      const float tot = xhalf_sum(acc[nt]);
      const int key = n0 + nt * 32 + r;
      const bool ok = key < p.Lk;
      if (csp && hh == 0) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)(csp + (int64_t)g * p.Lk), 0, p.Lk * 4, 0x00020000);
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, tot), rs, r * 4, (n0 + nt * 32) * 4, 0);
      }
      val[nt] = ok ? tot : 0.f;
      blk += val[nt];
      acc[nt] = 0.f;
    }
    flush_stores += (csp ? 2 : 0) + (bsp && n0 < p.Lk ? 1 : 0);
    if (bsp) {
      // Without the columns in memory the block sum is the caller's only view of them; it is then added up the way a
      // reduction over the stored columns adds (four neighbours in sequence, then a tree over the fours), so that
      // whoever ranks blocks gets the same ranking from either form.
      blk = csp ? group_sum<32>(blk) : quad_tree_sum(val[0]) + quad_tree_sum(val[1]);
      if (ln == 0 && n0 < p.Lk) bsp[(int64_t)g * p.nkb + kblk] = blk;
    }
  };

  const int kbase_l = r * ROWB + ((hh ^ ((r / SWD) & SWM)) << 4);
  float acc[2] = {0.f, 0.f};
  // the group being summed and the row of this range that it ends with (ranges begin with a group)
  int group = __builtin_amdgcn_readfirstlane(qoff / p.group_rows), group_end = p.group_rows;

  // probabilities of tile u from its logits: p = exp2(s*c - lse2[row]); rows >= Lq add nothing
  auto exp_acc = [&](int u, const f32x16& s0, const f32x16& s1) {
    const int hh = lane_id() >> 5;
    const char* ll = smem + LSE_OFF + ((u >> 1) & (NLSE - 1)) * 256 + ((u & 1) * 32 + 4 * hh) * 4;
    f32x4 lse[4];
#pragma unroll
    for (int j = 0; j < 4; j++) lse[j] = *(const f32x4*)(ll + j * 32);
    const bool ragged = (u * 32 + 32 > Lq_l);
    const int lim = Lq_l - u * 32 - 4 * hh;
    float pa = 0.f, pb = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      float x0 = fast_exp2(fmaf(s0[i], c, -lse[i >> 2][i & 3]));
      float x1 = fast_exp2(fmaf(s1[i], c, -lse[i >> 2][i & 3]));
      if (ragged) {
        const bool ok = (8 * (i >> 2) + (i & 3)) < lim;
        x0 = ok ? x0 : 0.f;
        x1 = ok ? x1 : 0.f;
      }
      pa += x0;
      pb += x1;
    }
    acc[0] += pa;
    acc[1] += pb;
    const int qend = u * 32 + 32;
    if (qend == group_end || qend >= Lq_l) flush(group, acc);
  };

  wait_fills(0);
  __syncthreads();

  const f32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};   // constant addend of the first MFMA
  // S(u) -> (n0a, n1a) on the matrix cores, nothing beside it
  auto qk_tile = [&](int u, f32x16& n0a, f32x16& n1a) {
    const char* qb = smem + ((u >> 1) & (NSTAGE - 1)) * QTILE + (u & 1) * 32 * ROWB;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      const bf16x8 f = *(const bf16x8*)(qb + (kbase_l ^ (ks << 5)));
      n0a = mfma32(f, kf[0][ks], ks == 0 ? zero : n0a);
      n1a = mfma32(f, kf[1][ks], ks == 0 ? zero : n1a);
    }
  };

  // One pipelined step: S(u) -> (n0, n1) on the matrix cores, probabilities of tile u-1 from (c0, c1)
  // on the vector ALU, interleaved by hand (sched_barrier(0) pins each group).
  auto step = [&](int u, f32x16& n0a, f32x16& n1a, const f32x16& c0, const f32x16& c1) {
    constexpr int AHEAD = 2;
    // The swizzled offsets of the KS reads are formed here, not kept in registers across the loop: from the address of the
    // stage (aligned beyond the bits that the swizzle changes), so that each costs one vector instruction, not two (six of
    // 117 per tile: 4096 x 10521 338.7 -> 335.3 us, 2304 x 6425 123.1 -> 121.7)
    int kb_l = kbase_l + (int)lds0 + ((u >> 1) & (NSTAGE - 1)) * QTILE;
    asm volatile("" : "+v"(kb_l));
    auto qread = [&](int j) -> bf16x8 { return *(LVAR_LDS const bf16x8*)(uintptr_t)(uint32_t)((kb_l ^ (j << 5)) + (u & 1) * 32 * ROWB); };
    bf16x8 frag[KS];
#pragma unroll
    for (int j = 0; j < AHEAD && j < KS; j++) frag[j] = qread(j);
    const int up = u - 1;
    const LVAR_LDS char* ll = (const LVAR_LDS char*)(uintptr_t)(lds0 + LSE_OFF + ((up >> 1) & (NLSE - 1)) * 256 + ((up & 1) * 32 + 4 * hh) * 4);
    // row statistics of four accumulator indices at a time, two reads ahead of their use (all four at once would cost
    // the registers of the third workgroup per compute unit)
    f32x4 lse[4];
    lse[0] = *(LVAR_LDS const f32x4*)ll;
    lse[1] = *(LVAR_LDS const f32x4*)(ll + 32);
    float pa = 0.f, pb = 0.f;
    // probabilities of tile u-1 as a three-stage pipeline over the MFMA steps (scale | exp2 | add), 16 / KS
    // accumulator indices of both key tiles per step, so that no vector instruction waits for the last one
    constexpr int EPS = 16 / KS;
    float xs0[16], xs1[16];
    auto st_scale = [&](int g) {
#pragma unroll
      for (int e = 0; e < EPS; e++) {
        const int i = g * EPS + e;
        xs0[i] = fmaf(c0[i], c, -lse[i >> 2][i & 3]);
        xs1[i] = fmaf(c1[i], c, -lse[i >> 2][i & 3]);
        if ((i & 3) == 3 && (i >> 2) + 2 < 4) lse[(i >> 2) + 2] = *(LVAR_LDS const f32x4*)(ll + ((i >> 2) + 2) * 32);
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
        pa += xs0[i];
        pb += xs1[i];
      }
    };
    st_scale(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      if (ks + AHEAD < KS) frag[ks + AHEAD] = qread(ks + AHEAD);
      n0a = mfma32(frag[ks], kf[0][ks], ks == 0 ? zero : n0a);
      n1a = mfma32(frag[ks], kf[1][ks], ks == 0 ? zero : n1a);
      if (ks >= 1) st_add(ks - 1);
      st_exp(ks);
      if (ks + 1 < KS) st_scale(ks + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    st_add(KS - 1);
    acc[0] += pa;
    acc[1] += pb;
    if (up * 32 + 32 == group_end) {
      flush(group, acc);
      group++;
      group_end += p.group_rows;
    }
  };

  // Tiles 0 .. U-2 go through the pipelined step (their successor exists); every tile whose rows are
  // all valid is consumed inside the next step, the last tile (possibly ragged) by exp_acc below.
  f32x16 sa0, sa1, sb0, sb1;
  qk_tile(0, sa0, sa1);
  for (int s = 0; s < S; s++) {
    flush_stores = 0;
    if (s > 0) {
      if (s + 1 < S) issue_stage(s + 1);   // into the stage that every wave has finished reading
      step(2 * s, sa0, sa1, sb0, sb1);
    }
    if (2 * s + 1 < U) step(2 * s + 1, sb0, sb1, sa0, sa1);
    wait_fills(flush_stores);
    __syncthreads();
  }
  // last tile U-1: in (sb) if U is even, else in (sa)
  if (U & 1) exp_acc(U - 1, sa0, sa1); else exp_acc(U - 1, sb0, sb1);
#endif  // __HIP_DEVICE_COMPILE__
}

template <int D, bool SOME>
static int launch_cs(const ColsumParams& p0, hipStream_t stream) {
  ColsumParams p = p0;
  if (p.kv_group < 1) p.kv_group = 1;
  p.nkb = (p.Lk + 63) / 64;
  p.nkt = (p.Lk + 255) / 256;
  // Ranges of query groups per key tile.  Workgroups are handed to the resident slots as slots
  // fall free, so a launch takes about its total work spread over the slots plus a part of the longest workgroup, during
  // which the chip drains.  More, shorter ranges shorten that tail and pay the fixed cost of a workgroup more often.
  // In 64-row stages, fitted to launches of 0.06 .. 0.37 ms on 256 compute units:
  //   cost = workgroups x (stages of a range + 1.5) / slots  +  0.4 x (stages of the longest range + 1.5)
  const int unit = (p.group_rows % 64 == 0) ? p.group_rows : (p.group_rows % 32 == 0 ? 2 * p.group_rows : 0);   // lcm(group_rows, 64)
  p.q_splits = 1;
  p.split_rows = ((p.Lq + 63) / 64) * 64 + (unit > 0 ? unit : 64);   // one range covers everything
  const int base_wg = p.B * p.H * p.nkt, slots = (D <= 128 ? CS_WGS : 1) * device_cus();
  if (unit > 0 && slots > 0 && base_wg < 4 * slots) {   // longer launches: the tail is small whatever the cut
    const int units_total = (p.Lq + unit - 1) / unit;
    double best = -1.0;
    for (int s = 1; s <= 8 && s <= units_total; s++) {
      const int rows = ((units_total + s - 1) / s) * unit;          // rows per range
      const int n = (p.Lq + rows - 1) / rows;                       // ranges that hold rows
      const int st_long = (std::min(rows, p.Lq) + 63) / 64, st_last = (p.Lq - (n - 1) * rows + 63) / 64;
      const double work = (double)base_wg * ((n - 1) * (st_long + 1.5) + (st_last + 1.5)) / slots;
      const double cost = work + 0.4 * (st_long + 1.5);
      if (best < 0.0 || cost < best) { best = cost; p.q_splits = n; p.split_rows = rows; }
    }
  }
  p.total_wg = base_wg * p.q_splits;
  const int grid = ((p.total_wg + 7) / 8) * 8;
  constexpr int SMEM = 2 * 64 * D * 2 + 4 * 256;
  static std::atomic<uint64_t> lds_ready{0};
  if (!ensure_lds_limit((const void*)colsum_kernel<D, SOME>, SMEM, lds_ready)) return LVAR_ELAUNCH;
  hipLaunchKernelGGL((colsum_kernel<D, SOME>), dim3(grid), dim3(256), SMEM, stream, p);
  return hipGetLastError() == hipSuccess ? LVAR_OK : LVAR_ELAUNCH;
}

int launch_colsum(const ColsumParams& p, int head_dim, hipStream_t s) {
  if (head_dim == 128) return p.some ? launch_cs<128, true>(p, s) : launch_cs<128, false>(p, s);
  if (head_dim == 64) return p.some ? launch_cs<64, true>(p, s) : launch_cs<64, false>(p, s);
  if (head_dim == 256) return p.some ? launch_cs<256, true>(p, s) : launch_cs<256, false>(p, s);
  return LVAR_EUNSUPPORTED;
}

}  // namespace lvar
