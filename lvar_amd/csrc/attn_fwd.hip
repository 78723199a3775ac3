// Flash-attention forward for gfx950 over a list of 64-key tiles: dense, block-list
// (flex BlockMask layout) and token-list (column-sparse, gathered keys) variants.
//
// Work decomposition
//   workgroup  = NWAVES waves, 32 query rows per wave (small launches: per two waves, see PAIR), all share the K/V tiles in LDS
//                (token lists with 192-row groups: 8 waves = 6 computing waves + 2 waves that only fetch, see NPROD; fewer rows
//                and four fetch waves in small launches; launch_forms.h says which launch takes which form)
//   wave       = S^T[64 keys x 32 queries] = K_tile . Q^T with 32x32x16 bf16 MFMA (K rows are
//                the A operand read from LDS, Q^T is the B operand held in registers), so a
//                lane owns ONE query column: the softmax row max / sum are in-register
//                reductions plus one exchange with lane^32.
//                O^T[d x 32 queries] += V^T . P^T: the S^T accumulators, packed to bf16, are
//                already in B-operand layout; V^T comes from the row-major V tile through
//                transposing LDS reads (ds_read_b64_tr_b16).
//   data path  = K/V rows go global -> LDS directly (buffer_load ... lds, 16 B per lane, no
//                register staging).  An instruction fills 1 KiB of consecutive LDS, so rows are
//                unpadded; bank conflicts are avoided by an XOR swizzle of the 16-byte chunk index
//                applied on the global side (each lane fetches the chunk that belongs in its slot).
//   pipeline   = iteration t issues the loads of K(t+2) and V(t+1); the matrix cores run
//                S(t+1) = K(t+1) Q^T and then O += P(t) V(t) while the vector ALU computes
//                P(t) = exp2(S(t)) and then the row maximum of S(t+1).  K and V are double-buffered,
//                one barrier per tile.
// Softmax runs in the exp2 domain with a lazily updated reference maximum: accumulators are
// rescaled only when some row maximum grows by more than RESCALE_TAU, which is exact
// because numerator and denominator share the same reference.
#include <type_traits>
#include "common.h"
#include "launch.h"
#include "launch_forms.h"
#include "sk_partition.h"

namespace lvar {

constexpr int READ_AHEAD = 4;    // operand fragments requested from LDS this many MFMAs before their use
constexpr int EXP_IN_QK = 24;    // of the 32 exp2 per lane and tile, how many run next to the QK MFMAs

// First S element of softmax slot g: EA elements spread over the NQK steps of the QK phase, the other
// 32 - EA over the first HB steps of the PV phase; slots before 0 and after the last one are empty.
template <int NQK, int HB, int EA>
struct ExpSlots {
  static constexpr int lo(int g) {
    return g <= 0 ? 0 : g < NQK ? g * EA / NQK : g < NQK + HB ? EA + (g - NQK) * (32 - EA) / (HB ? HB : 1) : 32;
  }
};

// The same for the 16 elements of a wave of a pair, over G slots
template <int G>
struct HalfSlots {
  static constexpr int lo(int g) { return g <= 0 ? 0 : g >= G ? 16 : g * 16 / G; }
};

// f(integral_constant<int, i>) for i = LO .. HI-1, unrolled at compile time
template <int LO, int HI, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (LO < HI) {
    f(std::integral_constant<int, LO>{});
    static_for<LO + 1, HI>(f);
  }
}
static constexpr float RESCALE_TAU = 8.0f;
static constexpr float NEG_BIG = -1.0e30f;

template <int D>
struct Swz {
  static constexpr int ROWB = D * 2;      // bytes per K/V row
  static constexpr int CPR = ROWB / 16;   // 16-byte chunks per row
  // chunk-index XOR of the K tile: makes ds_read_b128 of 16 consecutive rows conflict-free
  // (rows of 256 bytes or more: the row index itself, 16 rows per period)
  __device__ static __forceinline__ int fk(int row) {
    if constexpr (ROWB >= 256) return row & 15; else return (row / (256 / ROWB)) & (CPR - 1);
  }
  // chunk-index XOR of the V tile: moves the 64-byte segment read by the transposing loads of
  // 4 consecutive rows onto 4 different bank groups
  __device__ static __forceinline__ int fv(int row) { return (D >= 128) ? ((row & 3) << 2) : (((row >> 1) & 1) << 2); }
};

// Token-list instances whose list readers know two rows (AttnParams::remap_gs): 192-row groups in workgroups with fetch waves, or
// at head_dim 64 in two of three waves.  The others would pay the choice of a row per entry for nothing.
template <int D, int NWAVES, int MODE, int NPROD>
constexpr bool reads_remapped = MODE == MODE_GATHER && (NPROD > 0 || (D == 64 && NWAVES == 3));

// LDS of a workgroup: K and V buffers; the epilogue's transpose buffer of eight computing waves is larger.  Pairs of waves: behind
// the K and V buffers, two deep, every computing wave's half of P and one float per lane.
template <int D, int NCOMP, int MODE, bool PAIR = false>
constexpr int attn_lds_bytes() {
  const int bufs = 4 * 64 * D * 2, epi = NCOMP * 32 * (D * 2 + 16);
  if (PAIR) return bufs + 2 * NCOMP * (2048 + 256);
  return (MODE == MODE_BLOCK && epi > bufs) ? epi : bufs;
}

// Context of a balanced launch (see sk_partition.h); unused by the plain launch.
#if defined(__HIP_DEVICE_COMPILE__)
struct SkCtx {
  int slot0;        // workspace slot of piece 0 of this item's query tile
  int pieces;       // pieces of the tile (1 = whole)
  int kp;           // which piece this item is
  int tile_units;   // units of the whole tile
};

// Wait until at most N of this wave's global reads and LDS fills are outstanding (they complete in order)
template <int N>
__device__ __forceinline__ void wait_fills() {
  static_assert(N < 64, "six bits of the counter");
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));
}

// x, never fused with what is added to it: whether the compiler would depends on the instance, and all have the same bits
__device__ __forceinline__ float rounded(float x) {
  asm volatile("" : "+v"(x));
  return x;
}

// One query tile w (or, in a balanced launch, the units [u0, u1) of its tile list; `whole` = all of them).
//
// PAIR: two waves share 32 query rows, for launches that leave compute units idle: there a wave is alone on its SIMD and its chain
// of instructions per tile is the time of a tile (1800 .. 1900 cycles, 1066 of them MFMAs, however they are arranged).  Wave
// `half` of a pair forms S^T of keys 32 * half .. +31 of every tile, their softmax and their half of P, and accumulates columns
// half * D/2 .. of O over all 64 keys: half of the MFMAs and of the vector work each (1400 cycles).  P and the row maxima pass
// between the two through LDS behind the barrier that a tile has anyway: O is one tile behind S, so nothing in an iteration waits
// for anything else in it.  The order of every sum is the same as without: same bits.
template <int D, int NWAVES, int MODE, bool ACCUM, bool LSE_ONLY, bool SK, int NPROD, bool IDLE, bool PAIR = false, bool THIRD = false>
__device__ __forceinline__ void attn_item(const AttnParams& p, char* smem, const int w, const int bh, const int qt,
                                          const int u0, const int u1, const bool whole, const SkCtx& sk) {
  // NPROD: the last waves only fetch -- they read the list, form the addresses and issue every K/V fill -- and the
  // others compute.  Token lists with 8 waves: six compute (one 192-row group fills 6 of the 8 wave slots of a CU) and
  // two fetch, so the computing waves lose ~10 % of their instructions.  Launches of at most one 128-row workgroup per
  // CU: four and four (see fetch_waves).  Everywhere else all waves do both.
  constexpr int NCOMP = NWAVES - NPROD;     // computing waves, 32 query rows each
  constexpr int FW = NPROD ? NPROD : NWAVES;  // waves that issue the fills
  constexpr int RB = PAIR ? NCOMP / 2 : NCOMP;   // 32-row blocks
  constexpr int WGROWS = RB * 32;
  constexpr int KS = D / 16, MTD = D / 32;
  constexpr int MTW = PAIR ? MTD / 2 : MTD;      // 32-column blocks of O that a wave accumulates
  static_assert(!PAIR || (NPROD > 0 && !LSE_ONLY && !SK), "pairs have fetch waves beside them");
  constexpr int ROWB = Swz<D>::ROWB, CPR = Swz<D>::CPR;
  constexpr int RPI = 1024 / ROWB;          // rows filled by one 64-lane x 16 B load
  constexpr int NI = 64 / RPI;              // loads per 64-row tile
  constexpr int SLOTS = (NI + FW - 1) / FW;
  constexpr int TILE = 64 * ROWB;
  // block lists: the rows of a tile are consecutive, so a fill's lane offset can be a constant (see issue_slot)
  constexpr bool CONST_OFF = MODE == MODE_BLOCK && ((FW * RPI) % 16 == 0 || 16 % (FW * RPI) == 0) && NI % FW == 0;
  constexpr int CONST_PER = (FW * RPI) >= 16 ? 1 : 16 / (FW * RPI);
  constexpr int OSTR = D * 2 + 16;  // epilogue transpose buffer row stride (bytes)
  static_assert(RB * 32 * OSTR <= attn_lds_bytes<D, NCOMP, MODE, PAIR>(), "the epilogue buffer must fit");
  // LDS map: K buffers at 0 and TILE, V buffers at 2*TILE and 3*TILE

  const int b = bh / p.H, h = bh - b * p.H;
  const int tid = __builtin_amdgcn_workitem_id_x(), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = lane >> 5, r = lane & 31;
  const int half = (PAIR && wave >= RB) ? 1 : 0;   // which wave of a pair
  const int rblk = PAIR ? wave - half * RB : wave; // the block of 32 rows that it works on (fetch waves: no matter)
  const int fwave = NPROD ? wave - NCOMP : wave;   // index among the filling waves (negative: this wave does not fill)
  const int q0 = qt * WGROWS;
  const int g = q0 / p.group_rows;

  // Key-tile list of this query group.  Dense attention is the block-list variant with a null
  // list pointer, read as the identity list of ceil(Lk/64) 64-key blocks.
  const bool identity = (MODE == MODE_BLOCK) && p.list == nullptr;
  const int32_t* list = nullptr;
  int T, count;
  int tile0 = 0;   // identity list of a balanced launch: first tile of this piece
  int avail = 0;   // entries of the list row from `list` on (token lists)
  // Token lists formed from another scale's (see AttnParams): the waves that read the list take the entries straight from the
  // two rows they come from, so that no launch writes the lists and the count is not waited for.  Step at the last scale with
  // 20 % of the keys and a local run, B2 H16 d128: 30 x 30 32.8 -> 29.7 us, 48 x 48 84.5 -> 81.4; the whole 64 x 64
  // step 178.6 -> 176.2.
  constexpr bool REMAP = !SK && reads_remapped<D, NWAVES, MODE, NPROD>;
  int n_src = 0x7fffffff;             // entries from `list`, the others from `local`:
  const int32_t* local = nullptr;     // low words of 64-bit entries
  // first four entries of a block list, read together with the count (not after it): one memory
  // round trip less before the first tile can be fetched; entries beyond the count are never used
  int head[4] = {0, 0, 0, 0};
  if (identity) {
    count = (p.Lk + 63) >> 6;
    if (SK) { tile0 = u0; count = max(0, min(u1, count) - u0); }
    T = count;
  } else if (REMAP && p.remap_gs > 0) {
    const int gs = __builtin_amdgcn_readfirstlane(remap_group(g, p.remap_gk, p.remap_gs));
    list = p.list + b * p.list_sb + h * p.list_sh + (int64_t)gs * p.list_sg;
    local = (const int32_t*)(p.remap_local + (int64_t)g * p.remap_local_sg);
    n_src = p.remap_cnt;
    count = avail = n_src + p.remap_len;
    T = (count + 63) >> 6;
  } else {
    list = p.list + b * p.list_sb + h * p.list_sh + (int64_t)g * p.list_sg;
    const int first = SK ? (MODE == MODE_BLOCK ? u0 : (u0 << 6)) : 0;   // first list entry of this piece
    if (MODE == MODE_BLOCK) {
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (first + i < p.list_len) head[i] = list[first + i];
    }
    count = max(0, min(p.cnt[b * p.cnt_sb + h * p.cnt_sh + g], p.list_len));
    avail = p.list_len - first;
    if (SK) {
      const int last = (MODE == MODE_BLOCK) ? u1 : (u1 << 6);
      count = max(0, min(count, last) - first);
      list += first;
    }
    T = (MODE == MODE_BLOCK) ? (count << p.sub_shift) : ((count + 63) >> 6);
  }
  const int sub_shift = identity ? 0 : p.sub_shift;

  // accumulators and softmax state (one query column per lane pair l, l^32)
  f32x16 oacc[MTW];
#pragma unroll
  for (int m = 0; m < MTW; m++)
#pragma unroll
    for (int i = 0; i < 16; i++) oacc[m][i] = 0.f;
  float m_ref = NEG_BIG, m_true = -INFINITY;
  float lsum[2] = {0.f, 0.f};   // row sums of keys 0 .. 31 and of keys 32 .. 63 of every tile (what the two waves of a pair hold)
  const float c = p.c;

  if (T > 0) do {
    // raw buffer descriptors of this (batch, head) slice of K and V: base, stride 0, bound = the bytes of
    // the slice (below 2^31, checked on the host), so a fill beyond the last key row reads zeros
    auto make_rsrc = [](const void* base, int bytes) -> i32x4 {
      const uint64_t a = (uint64_t)base;
      i32x4 rs = {__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
                  __builtin_amdgcn_readfirstlane((int)(uint32_t)((a >> 32) & 0xffffu)),
                  __builtin_amdgcn_readfirstlane(bytes), 0x00020000};
      return rs;
    };
    const int k_srb = (int)p.k_sr * 2, v_srb = (int)p.v_sr * 2;  // row strides in bytes
    const int hkv = h / p.kv_group;   // grouped-query attention: kv_group query heads share a K/V head
    const i32x4 krsrc = make_rsrc(p.k + b * p.k_sb + hkv * p.k_sh, (p.Lk - 1) * k_srb + ROWB);
    const i32x4 vrsrc = make_rsrc(p.v + b * p.v_sb + hkv * p.v_sh, (p.Lk - 1) * v_srb + ROWB);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(LVAR_LDS char*)smem;

    // per-lane role in a tile load: row (within the RPI rows of one instruction) and chunk slot
    const int lrow = lane / CPR, lcs = lane % CPR;

    // Tile addressing is a two-step pipeline so that no list load is consumed in the iteration
    // that issued it: prefetch_raw(t) issues the list reads of tile t, finish_rows(t) turns them
    // (one iteration later) into a tile descriptor: for token lists the NR = SLOTS rows this lane
    // fetches, otherwise (NR = 1) the wave-uniform first row of the tile; plus nvalid = number of
    // leading tile rows that take part in the softmax.
    constexpr int NR = (MODE == MODE_GATHER) ? SLOTS : 1;
    auto prefetch_raw = [&](int t, int (&raw)[NR]) {
      if (MODE == MODE_BLOCK) {
        raw[0] = identity ? t + tile0 : list[t >> sub_shift];
      } else {
        // bounded by the row of the list, not by the count: entries behind the count are never used (they are
        // clamped and masked), and the read then does not have to wait for the count to arrive
#pragma unroll
        for (int s = 0; s < SLOTS; s++) {
          const int trow = (fwave + s * FW) * RPI + lrow;
          const int pos = (t << 6) + trow;
          const int32_t* e = list + pos;
          if constexpr (REMAP) e = pos < n_src ? e : local + 2 * (pos - n_src);
          raw[s] = (pos < avail && trow < 64) ? *e : 0;
        }
      }
    };
    auto finish_rows = [&](int t, const int (&raw)[NR], int (&rows)[NR], int& nvalid) {
      if (MODE == MODE_BLOCK) {
        // a block index outside the key range (a caller's mistake) is clamped before it is scaled
        const int blk = max(0, min(__builtin_amdgcn_readfirstlane(raw[0]), (p.Lk - 1) >> (6 + sub_shift)));
        rows[0] = ((blk << sub_shift) + (t & ((1 << sub_shift) - 1))) << 6;
        nvalid = max(0, min(64, p.Lk - rows[0]));
      } else {
        nvalid = min(64, count - (t << 6));
#pragma unroll
        for (int s = 0; s < NR; s++) rows[s] = max(0, min(raw[s], p.Lk - 1));   // clamped once, used by the K and the V fill
      }
    };
    // Issue the global->LDS loads of one tile (K or V) into the LDS buffer at byte address `dst`.
    // Written as inline assembly so that the compiler does not serialise later LDS reads of the
    // OTHER buffers behind these fills; completion is awaited with vmcnt(0) before the barrier.
    // issue_slot: the s-th of the SLOTS fill instructions this wave contributes to a tile; issue: all of them.
    // `left`: std::true_type, or (in a scalar register) the number of tiles from the current one on, and nothing is fetched
    // where that is less than three.  The skip is a branch inside the assembly: one that the compiler sees ends its basic
    // block, and it then moves the softmax instructions of the steps before, whose results are only used later, behind it
    // (every other tile ran its 16 QK MFMAs with no vector work beside them).  With two waves per SIMD the other wave covers
    // most of that: 4096 x 10521 in lists of 25 % 183.9 -> 182.5 us, d128 2304 x 6425 in 64 x 64 blocks 106.3 -> 104.8; with one,
    // d256 1600 x 4121 220.9 -> 217.3.
    auto issue_slot = [&](const i32x4& rsrc, int srb, bool is_v, const int (&rows)[NR], uint32_t dst, int s, auto left) {
      constexpr bool ALWAYS = std::is_same_v<decltype(left), std::true_type>;
      const int i = fwave + s * FW;
      if (!((NI % FW == 0) || i < NI)) return;
      const uint32_t m0v = dst + i * 1024;
      // Block lists, tile fully inside K/V: the rows of a tile are consecutive, so the per-lane byte
      // offset (row within the first instruction, swizzled chunk: the swizzle does not depend on the
      // slot) is a constant and tile and slot only move a scalar offset.
      // The buffer descriptor ends with the last key row, so the rows of a ragged last tile that lie beyond it read
      // as zeros (they are masked in the softmax); the first row is never negative (finish_rows clamps the block).
      // (The swizzle has a period of 16 rows: slots whose rows are a whole period apart share the lane offset.  When
      // the FW * RPI rows that the filling waves cover per slot are fewer than 16, CONST_PER such offsets alternate.)
      if constexpr (CONST_OFF) {
        const int row0 = __builtin_amdgcn_readfirstlane(rows[0]);  // wave-uniform for block lists
        const int trow0 = (fwave + (s % CONST_PER) * FW) * RPI + lrow;
        const int voff = trow0 * srb + ((lcs ^ (is_v ? Swz<D>::fv(trow0) : Swz<D>::fk(trow0))) << 4);
        const int soff = (row0 + (s / CONST_PER) * CONST_PER * FW * RPI) * srb;
        if constexpr (!ALWAYS) {
          asm volatile(
              "s_cmp_lt_i32 %4, 3\n\t"
              "s_cbranch_scc1 .Lno_fill%=\n\t"
              "s_mov_b32 m0, %0\n\t"
              "s_nop 0\n\t"
              "buffer_load_dwordx4 %1, %2, %3 offen lds\n"
              ".Lno_fill%=:"
              :
              : "s"(m0v), "v"(voff), "s"(rsrc), "s"(soff), "s"(left)
              : "memory", "scc");
          return;
        }
        asm volatile(
            "s_mov_b32 m0, %0\n\t"
            "s_nop 0\n\t"
            "buffer_load_dwordx4 %1, %2, %3 offen lds"
            :
            : "s"(m0v), "v"(voff), "s"(rsrc), "s"(soff)
            : "memory");
        return;
      }
      const int trow = i * RPI + lrow;
      const int chunk = lcs ^ (is_v ? Swz<D>::fv(trow) : Swz<D>::fk(trow));
      int voff;
      if (MODE == MODE_GATHER) {
        // token rows and row strides are below 2^24 (checked on the host): one full-rate 24-bit multiply-add
        voff = (int)(((unsigned)rows[s < NR ? s : 0] & 0xffffffu) * ((unsigned)srb & 0xffffffu) + (unsigned)(chunk * 16));
      } else {
        const int grow = max(0, min(rows[0] + trow, p.Lk - 1));
        voff = grow * srb + chunk * 16;
      }
      asm volatile(
          "s_mov_b32 m0, %0\n\t"
          "s_nop 0\n\t"
          "buffer_load_dwordx4 %1, %2, 0 offen lds"
          :
          : "s"(m0v), "v"(voff), "s"(rsrc)
          : "memory");  // m0 is scratch here: nothing else in this kernel keeps a value in it
    };
    auto issue = [&](const i32x4& rsrc, int srb, bool is_v, const int (&rows)[NR], uint32_t dst) {
#pragma unroll
      for (int s = 0; s < SLOTS; s++) issue_slot(rsrc, srb, is_v, rows, dst, s, std::true_type{});
    };

    // K(0), the oldest of the fills of the prologue, has landed: S(0) does not need V(0) and K(1), which are waited for
    // after it.  (Every filling wave issues at least NI / FW fills per tile.)  B2 H16 d128: 144 x 265 9.12 -> 8.83 us, 576 x 1497
    // 24.4 -> 24.2, sink + window lists at 48 x 48 57.0 -> 56.3; d64 B8 256 x 680 11.4 -> 11.3.
    auto wait_first = [&]() {
      constexpr int PER = NI / FW;
      if (T > 1) wait_fills<LSE_ONLY ? PER : 2 * PER>();
      else wait_fills<LSE_ONLY ? 0 : PER>();
    };

    // valid keys of tile t of a token list (only the last tile can be ragged)
    auto nvalid_gather = [&](int t) { return max(0, min(64, count - (t << 6))); };

    // tiles 0..3: block lists use the entries read next to the count
    auto first_raw = [&](int t, int (&raw)[NR]) {
      if (MODE == MODE_BLOCK && !identity) {
        const int e = t >> sub_shift;
        raw[0] = (e == 0) ? head[0] : (e == 1) ? head[1] : (e == 2) ? head[2] : head[3];
      } else {
        prefetch_raw(t, raw);
      }
    };

    // A computing wave of a ragged last query tile that owns no row does not compute: it keeps its part of the fills and
    // meets the barriers, so the waves with rows have the matrix cores and the LDS reads to themselves, and a launch at
    // the power limit keeps its clock (dense B2 H16 d128, 1600 x 4121 in 256-row tiles, an eighth of them padding: 111.7 ->
    // 106.5 us).  Where no wave has that role otherwise (IDLE, see idle_waves_pay) it is an instance of its own.
    const bool no_rows = !SK && (NPROD > 0 || IDLE) && q0 + rblk * 32 >= p.Lq;
    if ((NPROD > 0 && wave >= NCOMP) || no_rows) {
      // ---- fetch waves: the fill schedule of the loop below and nothing else; one barrier per tile ----
      const bool fills = !NPROD || wave >= NCOMP;
      int rows_u[NR], rows_v[NR], rows_k[NR], rows_n[NR], raw[NR], rows0[NR];   // rows_u: tile t (pairs)
      int nv_unused;
#pragma unroll
      for (int s = 0; s < NR; s++) { rows_u[s] = 0; rows_v[s] = 0; rows_k[s] = 0; rows_n[s] = 0; raw[s] = 0; }
      // the list entries of the first four tiles are requested together (one memory round trip, not one per tile)
      int raw0[NR], raw1[NR], raw2[NR];
      if (fills) {
        first_raw(0, raw0);
        first_raw(1, raw1);
        first_raw(2, raw2);
        first_raw(3, raw);
        finish_rows(0, raw0, rows0, nv_unused);
        finish_rows(1, raw1, rows_v, nv_unused);
        finish_rows(2, raw2, rows_k, nv_unused);
        issue(krsrc, k_srb, false, rows0, lds0);
        if (!LSE_ONLY) issue(vrsrc, v_srb, true, rows0, lds0 + 2 * TILE);
        if (T > 1) issue(krsrc, k_srb, false, rows_v, lds0 + TILE);
      }
      wait_first();
      __syncthreads();
      wait_fills<0>();
      __syncthreads();   // the computing waves have read K(0): its buffer may be refilled
      for (int t = 0; t + 1 < T; t++) {
        if (fills) {
          const int par = t & 1;
          if constexpr (PAIR) {
            if (t > 0) issue(vrsrc, v_srb, true, rows_u, lds0 + (2 + par) * TILE);
          } else if (!LSE_ONLY) {
            issue(vrsrc, v_srb, true, rows_v, lds0 + (3 - par) * TILE);
          }
          if (t + 2 < T) issue(krsrc, k_srb, false, rows_k, lds0 + par * TILE);
          if (t + 3 < T) finish_rows(t + 3, raw, rows_n, nv_unused);
          if (t + 4 < T) prefetch_raw(t + 4, raw);
        }
        wait_fills<0>();
        __syncthreads();
#pragma unroll
        for (int s = 0; s < NR; s++) { rows_u[s] = rows_v[s]; rows_v[s] = rows_k[s]; rows_k[s] = rows_n[s]; }
      }
      if constexpr (PAIR) {   // V of the last tile
        const int last = __builtin_amdgcn_readfirstlane(T - 1);
        if (fills && last > 0) issue(vrsrc, v_srb, true, rows_u, lds0 + (2 + (last & 1)) * TILE);
        wait_fills<0>();
        __syncthreads();
      }
      __syncthreads();   // the one after the last tile
      if (SK) break;     // a balanced launch has more barriers to meet below
      return;
    }

    // Q^T fragments stay in registers for the whole key loop
    const int qrow = min(q0 + rblk * 32 + r, p.Lq - 1);
    const bf16_t* qp = p.q + b * p.q_sb + h * p.q_sh + (int64_t)qrow * p.q_sr + hh * 8;
    bf16x8 qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) qf[ks] = *(const bf16x8*)(qp + ks * 16);

    // per-lane LDS read offsets (swizzled); K: row r (+32), chunk 2*ks+hh; V: see lds_read_tr
    const int kbase_l = r * ROWB + ((hh ^ Swz<D>::fk(r)) << 4);
    const int sq = (lane & 15) >> 2, sm = lane & 3;
    const int vbase_l = (4 * hh + sq) * ROWB + (((Swz<D>::fv(sq)) | (((lane >> 4) & 1) << 1) | (sm >> 1)) << 4) + (sm & 1) * 8;

    // S^T tile = K_tile . Q^T (16 MFMA for d = 128)
    auto qk_tile = [&](const char* kbuf, f32x16& s0, f32x16& s1) {
#pragma unroll
      for (int i = 0; i < 16; i++) { s0[i] = 0.f; s1[i] = 0.f; }
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        const char* a = kbuf + (kbase_l ^ (ks << 5));
        bf16x8 a0 = *(const bf16x8*)(a);
        bf16x8 a1 = *(const bf16x8*)(a + 32 * ROWB);
        s0 = mfma32(a0, qf[ks], s0);
        s1 = mfma32(a1, qf[ks], s1);
      }
    };
    // keys beyond nvalid do not take part (only the last tile of a list can be ragged)
    auto mask_tile = [&](f32x16& s0, f32x16& s1, int nvalid) {
      // accumulator i of this lane is tile row 8*(i/4) + 4*hh + (i%4): compare against a per-lane
      // limit so that the per-element constants stay immediates
      const int lim = nvalid - 4 * hh;
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int kc = 8 * (i >> 2) + (i & 3);
        s0[i] = (kc < lim) ? s0[i] : -INFINITY;
        s1[i] = (kc + 32 < lim) ? s1[i] : -INFINITY;
      }
    };
    // row maximum of the raw logits of one tile (both lane halves)
    auto max_tile = [&](const f32x16& s0, const f32x16& s1) -> float {
      float ma = fmaxf(s0[0], s1[0]), mb = fmaxf(s0[1], s1[1]);
#pragma unroll
      for (int i = 2; i < 16; i += 2) {
        ma = fmaxf(fmaxf(ma, s0[i]), s1[i]);
        mb = fmaxf(fmaxf(mb, s0[i + 1]), s1[i + 1]);
      }
      return xhalf_max(fmaxf(ma, mb));
    };
    // lazy reference-maximum update for a tile whose raw row maximum is mx
    auto rescale_check = [&](float mx) {
      const float mt = mx * c;
      m_true = fmaxf(m_true, mt);
      if (__builtin_amdgcn_ballot_w64(mt > m_ref + RESCALE_TAU) != 0) {
        const float m_new = fmaxf(m_ref, mt);
        const float alpha = fast_exp2(m_ref - m_new);
        lsum[0] = rounded(lsum[0] * alpha);
        lsum[1] = rounded(lsum[1] * alpha);
        if (!LSE_ONLY) {
#pragma unroll
          for (int m = 0; m < MTD; m++)
#pragma unroll
            for (int i = 0; i < 16; i++) oacc[m][i] *= alpha;
        }
        m_ref = m_new;
      }
    };
    // P = exp2(S*c - m_ref), row-sum partials, bf16 pack into the B-operand layout of the PV MFMA
    auto exp_tile = [&](f32x16& s0, f32x16& s1, bf16x8 (&pb)[4]) {
      const float negm = -m_ref;
      float la = 0.f, lb = 0.f;
#pragma unroll
      for (int i = 0; i < 16; i++) {
        s0[i] = fast_exp2(fmaf(s0[i], c, negm));
        s1[i] = fast_exp2(fmaf(s1[i], c, negm));
        la += s0[i];
        lb += s1[i];
      }
      lsum[0] += la;
      lsum[1] += lb;
      pb[0] = pack8(s0[0], s0[1], s0[2], s0[3], s0[4], s0[5], s0[6], s0[7]);
      pb[1] = pack8(s0[8], s0[9], s0[10], s0[11], s0[12], s0[13], s0[14], s0[15]);
      pb[2] = pack8(s1[0], s1[1], s1[2], s1[3], s1[4], s1[5], s1[6], s1[7]);
      pb[3] = pack8(s1[8], s1[9], s1[10], s1[11], s1[12], s1[13], s1[14], s1[15]);
    };
    // O^T += V^T . P^T (16 MFMA for d = 128)
    auto pv_tile = [&](const bf16x8 (&pb)[4], const char* vbuf) {
#pragma unroll
      for (int kb = 0; kb < 4; kb++) {
#pragma unroll
        for (int m = 0; m < MTD; m++) {
          const char* a = vbuf + (vbase_l ^ (m << 6)) + kb * 16 * ROWB;
          bf16x4 lo = lds_read_tr(a);
          bf16x4 hi = lds_read_tr(a + 8 * ROWB);
          bf16x8 av = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
          oacc[m] = mfma32(av, pb[kb], oacc[m]);
        }
      }
    };

    // ---- prologue: tiles 0 and 1 in flight, S(0) computed ----
    // rows_v: rows of tile t+1 (its V is fetched next), rows_k: rows of tile t+2 (its K is next),
    // rows_n: rows of tile t+3, raw: list reads of tile t+4
    int rows_v[NR], rows_k[NR], rows_n[NR], raw[NR];
#pragma unroll
    for (int s = 0; s < NR; s++) { rows_v[s] = 0; rows_k[s] = 0; rows_n[s] = 0; raw[s] = 0; }
    int nv0, nv1 = 64, nv2 = 64, nv3 = 64;
    if constexpr (NPROD && MODE == MODE_GATHER) {
      nv0 = nvalid_gather(0); nv1 = nvalid_gather(1); nv2 = nvalid_gather(2);
    } else {
      int rows0[NR];
      if constexpr (MODE == MODE_GATHER) {
        // the list entries of the first four tiles are requested together (one memory round trip, not one per tile)
        int raw0[NR], raw1[NR], raw2[NR];
        prefetch_raw(0, raw0);
        prefetch_raw(1, raw1);
        prefetch_raw(2, raw2);
        prefetch_raw(3, raw);
        finish_rows(0, raw0, rows0, nv0);
        finish_rows(1, raw1, rows_v, nv1);
        finish_rows(2, raw2, rows_k, nv2);
        nv1 = max(nv1, 0); nv2 = max(nv2, 0);
      } else {
        first_raw(0, raw);
        finish_rows(0, raw, rows0, nv0);
        if (T > 1) { first_raw(1, raw); finish_rows(1, raw, rows_v, nv1); }
        if (T > 2) { first_raw(2, raw); finish_rows(2, raw, rows_k, nv2); }
        if (T > 3) first_raw(3, raw);
      }
      if constexpr (!NPROD) {
        issue(krsrc, k_srb, false, rows0, lds0);
        if (!LSE_ONLY) issue(vrsrc, v_srb, true, rows0, lds0 + 2 * TILE);
        if (T > 1) issue(krsrc, k_srb, false, rows_v, lds0 + TILE);
      }
    }
    if constexpr (NPROD) wait_fills<0>(); else wait_first();
    __syncthreads();
    if constexpr (PAIR) {
      char* const pbuf = smem + 4 * TILE;                        // [parity][row block][quarter of the keys][lane] x 16 bytes
      constexpr int PPAR = NCOMP * 2048;                         // bytes of one parity
      float* const xbuf = (float*)(pbuf + 2 * PPAR);             // [parity][computing wave][lane]
      const int mate = half ? wave - RB : wave + RB;
      int kb_l = kbase_l + half * 32 * ROWB;
      int vb_l[MTW];
#pragma unroll
      for (int m = 0; m < MTW; m++) vb_l[m] = vbase_l ^ ((half * MTW + m) << 6);
      char* const pmine = pbuf + (rblk * 4 + half * 2) * 1024 + lane * 16;
      const char* const prow = pbuf + rblk * 4096 + lane * 16;
      const int tiles = __builtin_amdgcn_readfirstlane(T);
      f32x16 sa, sb;
      float mown, alpha = 1.f;
      bool pend = false;
      auto kread = [&](const char* kbuf, int j) -> bf16x8 { return *(const bf16x8*)(kbuf + (kb_l ^ (j << 5))); };
      auto vread = [&](const char* vbuf, int j) -> bf16x8 {
        const char* a = vbuf + vb_l[j % MTW] + (j / MTW) * 16 * ROWB;
        bf16x4 lo = lds_read_tr(a);
        bf16x4 hi = lds_read_tr(a + 8 * ROWB);
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      };
      auto mask_half = [&](f32x16& x, int nvalid) {
        const int lim = nvalid - 32 * half - 4 * hh;
#pragma unroll
        for (int i = 0; i < 16; i++) x[i] = (8 * (i >> 2) + (i & 3) < lim) ? x[i] : -INFINITY;
      };
      auto max_half = [&](const f32x16& x) -> float {
        float a = fmaxf(x[0], x[1]);
#pragma unroll
        for (int i = 2; i < 16; i += 2) a = fmaxf(fmaxf(a, x[i]), x[i + 1]);
        return xhalf_max(a);
      };
      // the reference maximum of tile t, from the row maxima of both waves; O lacks P(t-1) V(t-1) yet, so its factor waits (pend)
      auto settle = [&](float mx) {
        const float mt = mx * c;
        m_true = fmaxf(m_true, mt);
        pend = __builtin_amdgcn_ballot_w64(mt > m_ref + RESCALE_TAU) != 0;
        if (pend) {
          const float m_new = fmaxf(m_ref, mt);
          alpha = fast_exp2(m_ref - m_new);
          lsum[0] = rounded(lsum[0] * alpha);
          m_ref = m_new;
        }
      };
      // Iteration t: the matrix cores run S(t+1) = K(t+1) Q^T (this wave's keys; hasqk) and O += P(t-1) V(t-1) (its columns; haspv)
      // while the vector ALU turns S(t) into P(t); K(t+1) is in K buffer 1 - PAR, V(t-1) in V buffer 1 - PAR.
      auto half_tile = [&](int t, auto par, auto masked, auto hasqk, auto haspv, f32x16& cs, f32x16& ns) {
        const int PAR = par;
        constexpr bool MASKED = decltype(masked)::value, QK = decltype(hasqk)::value, PV = decltype(haspv)::value;
        constexpr int NQK = QK ? KS : 0, NPV = PV ? 4 * MTW : 0, NS = NQK + NPV, AHEAD = READ_AHEAD, PAHEAD = 3;
        // the maximum is settled two MFMAs into the iteration: the other wave's arrives from LDS with the first fragments
        constexpr int CHK = NS >= 8 ? 2 : 0;
        using Sch = HalfSlots<(NS - CHK > 3 ? NS - CHK - 2 : 1)>;
        if constexpr (MODE == MODE_GATHER) {
          nv3 = nvalid_gather(t + 3);
        } else if constexpr (QK) {
          if (t + 3 < tiles) finish_rows(t + 3, raw, rows_n, nv3);
          if (t + 4 < tiles) prefetch_raw(t + 4, raw);
        }
        const char* kbuf = smem + (1 - PAR) * TILE;
        const char* vbuf = smem + (3 - PAR) * TILE;
        const float mother = xbuf[(PAR * NCOMP + mate) * 64 + lane];
        bf16x8 frag[NS > 0 ? NS : 1], pb[4];
        auto operand = [&](auto ic) {
          constexpr int i = decltype(ic)::value;
          if constexpr (i < NQK) frag[i] = kread(kbuf, i); else frag[i] = vread(vbuf, i - NQK);
        };
        // quarter kb of P(t-1), PAHEAD steps ahead of its first use
        auto p_operand = [&](auto ic) {
          constexpr int i = decltype(ic)::value - NQK + PAHEAD;
#pragma unroll
          for (int kb = 0; kb < 4; kb++)
            if (PV && (kb * MTW == i || (decltype(ic)::value == 0 && kb * MTW < i))) pb[kb] = *(const bf16x8*)(prow + (1 - PAR) * PPAR + kb * 1024);
        };
        uint32_t pw[8];
        float ls = 0.f, negm = 0.f, ma = -INFINITY;
        auto softmax_step = [&](auto gc) {
          constexpr int g = decltype(gc)::value;
          static_for<Sch::lo(g - 2), Sch::lo(g - 1)>([&](auto ec) {
            constexpr int e = decltype(ec)::value;
            ls += cs[e];
            if constexpr (e & 1) pw[e >> 1] = pack_bf16(cs[e - 1], cs[e]);
            if constexpr (e == 7 || e == 15) {
              const u32x4 u = {pw[(e >> 1) - 3], pw[(e >> 1) - 2], pw[(e >> 1) - 1], pw[e >> 1]};
              *(u32x4*)(pmine + PAR * PPAR + (e >> 3) * 1024) = u;
            }
          });
          static_for<Sch::lo(g - 1), Sch::lo(g)>([&](auto ec) { constexpr int e = decltype(ec)::value; cs[e] = fast_exp2(cs[e]); });
          static_for<Sch::lo(g), Sch::lo(g + 1)>([&](auto ec) { constexpr int e = decltype(ec)::value; cs[e] = fmaf(cs[e], c, negm); });
        };
        static_for<0, (AHEAD < NS ? AHEAD : NS)>(operand);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (CHK == 0) { settle(fmaxf(mown, mother)); negm = -m_ref; }
        static_for<0, NS>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          if constexpr (CHK > 0 && i == CHK) { settle(fmaxf(mown, mother)); negm = -m_ref; }
          if constexpr (i + AHEAD < NS) operand(std::integral_constant<int, i + AHEAD>{});
          p_operand(ic);
          if constexpr (i >= NQK) oacc[(i - NQK) % MTW] = mfma32(frag[i], pb[(i - NQK) / MTW], oacc[(i - NQK) % MTW]);
          else if constexpr (i == 0) ns = mfma32(frag[0], qf[0], f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0});
          else ns = mfma32(frag[i], qf[i], ns);
          if constexpr (i >= CHK) softmax_step(std::integral_constant<int, i - CHK>{});
          // row maximum of S(t+1), next to the PV steps
          if constexpr (QK && PV && i > NQK + 1) {
            if constexpr (MASKED && i == NQK + 2) mask_half(ns, nv1);
            constexpr int n = NPV - 2, k = i - NQK - 2;
#pragma unroll
            for (int e = k * 8 / n; e < (k + 1) * 8 / n; e++) ma = fmaxf(fmaxf(ma, ns[2 * e]), ns[2 * e + 1]);
          }
          __builtin_amdgcn_sched_barrier(0);
        });
        static_for<NS - CHK, 16 + 3>(softmax_step);   // what is left of the softmax
        lsum[0] += ls;
        if constexpr (PV) {
          if (pend) {
#pragma unroll
            for (int m = 0; m < MTW; m++)
#pragma unroll
              for (int i = 0; i < 16; i++) oacc[m][i] *= alpha;
          }
        }
        if constexpr (QK && PV) mown = xhalf_max(ma);
        if constexpr (QK && !PV) {
          if constexpr (MASKED) mask_half(ns, nv1);
          mown = max_half(ns);
        }
        xbuf[((1 - PAR) * NCOMP + wave) * 64 + lane] = QK ? mown : lsum[0];   // behind the last tile the row sums change hands
        __syncthreads();
        nv1 = nv2; nv2 = nv3;
#pragma unroll
        for (int s = 0; s < NR; s++) { rows_v[s] = rows_k[s]; rows_k[s] = rows_n[s]; }
      };
#pragma unroll
      for (int i = 0; i < 16; i++) sa[i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ks++) sa = mfma32(kread(smem, ks), qf[ks], sa);
      if (nv0 < 64) mask_half(sa, nv0);
      mown = max_half(sa);
      xbuf[wave * 64 + lane] = mown;
      __syncthreads();   // all have read K(0), and V(0) and K(1) have landed
      using P0 = std::integral_constant<int, 0>;
      using P1 = std::integral_constant<int, 1>;
      using Yes = std::true_type;
      using No = std::false_type;
      auto step = [&](int t, auto par, auto haspv, f32x16& cs, f32x16& ns) {
        if (nv1 < 64) half_tile(t, par, Yes{}, Yes{}, haspv, cs, ns);
        else half_tile(t, par, No{}, Yes{}, haspv, cs, ns);
      };
      // The last tile, of either parity: as two instances behind a branch O was held twice, for the path not taken, too, and at
      // head_dim 256 an even number of tiles spilled 36 registers on its way out (2 tiles 11.0 -> 8.3 us, 24 31.9 -> 28.2).
      auto last = [&](int par, auto haspv, f32x16& cs, f32x16& ns) {
        half_tile(tiles - 1, par, No{}, No{}, haspv, cs, ns);
        lsum[1] = xbuf[((1 - par) * NCOMP + mate) * 64 + lane];
#pragma unroll
        for (int kb = 0; kb < 4; kb++) {
          const bf16x8 pq = *(const bf16x8*)(prow + par * PPAR + kb * 1024);
#pragma unroll
          for (int m = 0; m < MTW; m++) oacc[m] = mfma32(vread(smem + (2 + par) * TILE, kb * MTW + m), pq, oacc[m]);
        }
        __syncthreads();
      };
      if (tiles == 1) {
        last(0, No{}, sa, sb);
        break;
      }
      step(0, P0{}, No{}, sa, sb);
      int t = 1;
      for (; t + 2 < tiles; t += 2) {
        step(t, P1{}, Yes{}, sb, sa);
        step(t + 1, P0{}, Yes{}, sa, sb);
      }
      if (t + 1 < tiles) step(t, P1{}, Yes{}, sb, sa);
      else sa = sb;
      last((tiles - 1) & 1, Yes{}, sa, sb);
      break;
    } else {
    f32x16 sa0, sa1, sb0, sb1;
    qk_tile(smem, sa0, sa1);
    // K(2) is fetched into the buffer of K(0) at the top of the first iteration: every wave must have read
    // K(0) before any wave issues that fill; and V(0) and K(1) have landed
    wait_fills<0>();
    __syncthreads();
    if (nv0 < 64) mask_tile(sa0, sa1, nv0);
    rescale_check(max_tile(sa0, sa1));

    // Pipelined iteration for a tile t that has a successor; PAR = t & 1 picks the buffers:
    //   K(t+1) is in K buffer (1-PAR), K(t+2) goes to K buffer PAR,
    //   V(t) is in V buffer PAR, V(t+1) goes to V buffer (1-PAR).
    // Between the two barriers the body is one straight-line block: the matrix cores run
    // S(t+1) = K(t+1) Q^T and then O += P(t) V(t) while the vector ALU turns S(t) into P(t) and
    // then reduces the row maximum of S(t+1); the reference-maximum update (a rare branch)
    // sits after the barrier.
    auto body = [&](int t, auto par, auto masked, f32x16& c0, f32x16& c1, f32x16& n0, f32x16& n1) {
      constexpr int PAR = decltype(par)::value;
      constexpr bool MASKED = decltype(masked)::value;
      // The fills of V(t+1) and K(t+2) are not issued in one burst up front (a wave spends tens of cycles on each and
      // the matrix cores would sit idle meanwhile) but one by one between the QK MFMAs, where their issue runs in the
      // shadow of the MFMA before.  NFILL instructions, one every FSTRIDE steps; if there are more than steps, up front.
      constexpr int NQK_ = 2 * KS;
      constexpr int NFILL = NPROD ? 0 : (LSE_ONLY ? SLOTS : 2 * SLOTS);
      constexpr int FSTRIDE = (CONST_OFF && NFILL > 0 && NFILL <= NQK_) ? NQK_ / NFILL : 0;
      // K(t+2) is only fetched if there is one.  The skip is inside the fill (see issue_slot) where fills are spread over the steps, but
      // not in the instance of three workgroups per compute unit: its third wave covers a branch, its registers are limited, and the
      // assembly's operands had 21 of them spilled (B3 H24 1024 x 1100 36.2 us, 33.6 with the branch; 10 % of 128 x 128 blocks at
      // 4096 x 10521 48.0, 43.9).  Fills in one burst up front (token lists) keep the branch, too, on T itself: on a copy of it in a
      // scalar register the 64-row groups of head_dim 128 spilled 69 registers, now 21 (4096 x 10521, 832 keys 210 / 137 us; 96-row
      // groups 154 / 117).
      constexpr bool SKIP_IN_FILL = FSTRIDE > 0 && !THIRD;
      const int left = SKIP_IN_FILL ? __builtin_amdgcn_readfirstlane(T - t) : 0;   // tiles from this one on
      const bool fill_k = t + 2 < T;
      auto fill_step = [&](auto jc) {
        constexpr int j = decltype(jc)::value;
        if constexpr (FSTRIDE > 0) {
          if constexpr (j % FSTRIDE == 0 && j / FSTRIDE < NFILL) {
            constexpr int f = j / FSTRIDE;
            if constexpr (!LSE_ONLY && f < SLOTS) issue_slot(vrsrc, v_srb, true, rows_v, lds0 + (3 - PAR) * TILE, f, std::true_type{});
            else if constexpr (SKIP_IN_FILL) issue_slot(krsrc, k_srb, false, rows_k, lds0 + PAR * TILE, LSE_ONLY ? f : f - SLOTS, left);
            else if (fill_k) issue_slot(krsrc, k_srb, false, rows_k, lds0 + PAR * TILE, LSE_ONLY ? f : f - SLOTS, std::true_type{});
          }
        }
      };
      if constexpr (NPROD && MODE == MODE_GATHER) {
        nv3 = nvalid_gather(t + 3);
      } else {
        if constexpr (!NPROD && FSTRIDE == 0) {
          if (!LSE_ONLY) issue(vrsrc, v_srb, true, rows_v, lds0 + (3 - PAR) * TILE);
          if (fill_k) issue(krsrc, k_srb, false, rows_k, lds0 + PAR * TILE);
        }
        if (t + 3 < T) finish_rows(t + 3, raw, rows_n, nv3);
        if (t + 4 < T) prefetch_raw(t + 4, raw);
      }
      // The block below is software-pipelined by hand; sched_barrier(0) after every step stops the
      // compiler from regrouping it.  Phase A: QK MFMA j | K-fragment read j+4 | softmax slot j of
      // S(t).  Phase B: PV MFMA j | the two transposing V reads of MFMA j+4 | the last softmax slots
      // of S(t) (first half) or a slice of the row-maximum reduction of S(t+1) (second half).
      constexpr int NQK = 2 * KS, NPV = LSE_ONLY ? 0 : 4 * MTD, AHEAD = READ_AHEAD;
      const char* kbuf = smem + (1 - PAR) * TILE;
      const char* vbuf = smem + (2 + PAR) * TILE;
      auto kread = [&](int j) -> bf16x8 {
        return *(const bf16x8*)(kbuf + (kbase_l ^ ((j >> 1) << 5)) + (j & 1) * 32 * ROWB);
      };
      auto vread = [&](int j) -> bf16x8 {
        const int kb = j / MTD, m = j % MTD;
        const char* a = vbuf + (vbase_l ^ (m << 6)) + kb * 16 * ROWB;
        bf16x4 lo = lds_read_tr(a);
        bf16x4 hi = lds_read_tr(a + 8 * ROWB);
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      };
      bf16x8 frag[NQK > NPV ? NQK : NPV];
      uint32_t pw[16];
      const float negm = -m_ref;
      // A half's sum joins the row sum as soon as it is complete: held to the end of the tile, the two cost a register more while the
      // V fragments and P need theirs (64- and 96-row token-list groups at head_dim 128 spill 14 and 0 registers, not 21 and 19:
      // 4096 x 10521, 832 keys 137 / 133 and 117 / 95 us; the statistics at head_dim 64 keep to 128, four waves per SIMD: 4096 x 10521
      // 266 / 260).  Where registers are to spare the chain of additions is better split: the other instances of head_dim 64 lose 1 %
      // of their lists' time with it, the statistics at head_dim 128 (up to 2 %, 130 x 147 5.37 / 5.50) and 256 1.5 %.
      constexpr bool SUM_EARLY = LSE_ONLY ? D == 64 : D > 64 || THIRD;
      float la = 0.f, lb = 0.f;
      // The softmax of S(t) runs as a three-stage pipeline over the MFMA steps so that no vector instruction
      // waits for the one before it: step g scales the elements of slot g, takes exp2 of slot g-1 and
      // adds / packs slot g-2.  Slots: EA elements over the QK steps, the rest over the first half of the
      // PV steps (quarter kb of P is complete before PV step kb * MTD needs it); the row maximum of
      // S(t+1) goes next to the second half of the PV steps.
      auto st_scale = [&](auto ec) {
        constexpr int e = decltype(ec)::value;
        if constexpr (e < 16) c0[e] = fmaf(c0[e], c, negm); else c1[e - 16] = fmaf(c1[e - 16], c, negm);
      };
      auto st_exp = [&](auto ec) {
        constexpr int e = decltype(ec)::value;
        if constexpr (e < 16) c0[e] = fast_exp2(c0[e]); else c1[e - 16] = fast_exp2(c1[e - 16]);
      };
      auto st_sum = [&](auto ec) {
        constexpr int e = decltype(ec)::value;
        float r;
        if constexpr (e < 16) r = c0[e]; else r = c1[e - 16];
        if constexpr (e < 16) la += r; else lb += r;
        if constexpr (SUM_EARLY && e == 15) lsum[0] += la;
        if constexpr (SUM_EARLY && e == 31) lsum[1] += lb;
        if constexpr (e & 1) {
          float prev;
          if constexpr (e < 16) prev = c0[e - 1]; else prev = c1[e - 17];
          pw[e >> 1] = pack_bf16(prev, r);
        }
      };
      using Sch = ExpSlots<2 * KS, (LSE_ONLY ? 0 : 4 * MTD) / 2, LSE_ONLY ? 32 : EXP_IN_QK>;
      auto softmax_step = [&](auto gc) {
        constexpr int g = decltype(gc)::value;
        static_for<Sch::lo(g - 2), Sch::lo(g - 1)>(st_sum);
        static_for<Sch::lo(g - 1), Sch::lo(g)>(st_exp);
        static_for<Sch::lo(g), Sch::lo(g + 1)>(st_scale);
      };
      constexpr int HB = NPV / 2;
#pragma unroll
      for (int j = 0; j < AHEAD; j++) frag[j] = kread(j);
      __builtin_amdgcn_sched_barrier(0);
      static_for<0, NQK>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        if constexpr (j + AHEAD < NQK) frag[j + AHEAD] = kread(j + AHEAD);
        // the first MFMA of each accumulator takes the constant 0 as its addend (no register clearing)
        if constexpr (j == 0) n0 = mfma32(frag[j], qf[0], f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0});
        else if constexpr (j == 1) n1 = mfma32(frag[j], qf[0], f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0});
        else if constexpr (j & 1) n1 = mfma32(frag[j], qf[j >> 1], n1);
        else n0 = mfma32(frag[j], qf[j >> 1], n0);
        fill_step(jc);
        softmax_step(jc);
        __builtin_amdgcn_sched_barrier(0);
      });
      float ma = -INFINITY, mb = -INFINITY;
      if (!LSE_ONLY) {
        bf16x8 pb[4];
#pragma unroll
        for (int j = 0; j < AHEAD; j++) frag[j] = vread(j);
        __builtin_amdgcn_sched_barrier(0);
        if (MASKED) mask_tile(n0, n1, nv1);
        static_for<0, NPV>([&](auto jc) {
          constexpr int j = decltype(jc)::value;
          if constexpr (j + AHEAD < NPV) frag[j + AHEAD] = vread(j + AHEAD);
          if constexpr (j % MTD == 0) {
            constexpr int kb = j / MTD;
            u32x4 u = {pw[4 * kb], pw[4 * kb + 1], pw[4 * kb + 2], pw[4 * kb + 3]};
            pb[kb] = __builtin_bit_cast(bf16x8, u);
          }
          oacc[j % MTD] = mfma32(frag[j], pb[j / MTD], oacc[j % MTD]);
          softmax_step(std::integral_constant<int, NQK + j>{});
          if constexpr (j >= HB) {
            constexpr int e0 = (j - HB) * 16 / (NPV - HB), e1 = (j - HB + 1) * 16 / (NPV - HB);
#pragma unroll
            for (int e = e0; e < e1; e++) ma = fmaxf(fmaxf(ma, n0[e]), n1[e]);
          }
          __builtin_amdgcn_sched_barrier(0);
        });
      } else {
        softmax_step(std::integral_constant<int, NQK>{});
        softmax_step(std::integral_constant<int, NQK + 1>{});
        if (MASKED) mask_tile(n0, n1, nv1);
#pragma unroll
        for (int e = 0; e < 16; e++) ma = fmaxf(fmaxf(ma, n0[e]), n1[e]);
      }
      if constexpr (!SUM_EARLY) {
        lsum[0] += la;
        lsum[1] += lb;
      }
      const float mx = xhalf_max(fmaxf(ma, mb));
      wait_fills<0>();
      __syncthreads();
      rescale_check(mx);
      nv0 = nv1; nv1 = nv2; nv2 = nv3;
      if constexpr (!(NPROD && MODE == MODE_GATHER)) {
#pragma unroll
        for (int s = 0; s < NR; s++) { rows_v[s] = rows_k[s]; rows_k[s] = rows_n[s]; }
      }
    };
    auto step = [&](int t, auto par, f32x16& c0, f32x16& c1, f32x16& n0, f32x16& n1) {
      if (nv1 < 64) body(t, par, std::true_type{}, c0, c1, n0, n1);
      else body(t, par, std::false_type{}, c0, c1, n0, n1);
    };
    // last tile of the list: no successor to prefetch or to multiply
    auto last = [&](auto par, f32x16& c0, f32x16& c1) {
      constexpr int PAR = decltype(par)::value;
      bf16x8 pb[4];
      exp_tile(c0, c1, pb);
      if (!LSE_ONLY) pv_tile(pb, smem + (2 + PAR) * TILE);
      __syncthreads();
    };

    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    int t = 0;
    for (; t + 2 < T; t += 2) {
      step(t, P0{}, sa0, sa1, sb0, sb1);
      step(t + 1, P1{}, sb0, sb1, sa0, sa1);
    }
    if (t + 1 < T) {
      step(t, P0{}, sa0, sa1, sb0, sb1);
      last(P1{}, sb0, sb1);
    } else {
      last(P0{}, sa0, sa1);
    }
    }
  } while (false);

  if constexpr (SK) {
    if (!whole) {
      // ---- a piece of a query tile: park the unnormalised state in the piece's workspace slot; the workgroup
      // whose piece completes the tile adds all pieces up, in list order, and runs the epilogue ----
      constexpr int SLOT_FLOATS = D * 32 * NCOMP + 3 * 64 * NCOMP;
      const bool computes = !(NPROD && wave >= NCOMP);
      // The pieces travel between XCDs, whose L2 caches do not see each other's lines.  Rather than writing back
      // and invalidating whole caches around the exchange (what device-scope fences do), every workspace access is
      // itself device-coherent: relaxed device-scope atomic stores and loads write through / read past the L2.  The
      // stores are awaited before the arrival counter is bumped, the loads are issued after its value came back.
      auto put2 = [](float* dst, float a, float b) {
        const uint64_t v = (uint64_t)__builtin_bit_cast(uint32_t, a) | ((uint64_t)__builtin_bit_cast(uint32_t, b) << 32);
        __hip_atomic_store((uint64_t*)dst, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      };
      auto get2 = [](const float* src, float& a, float& b) {
        const uint64_t v = __hip_atomic_load((const uint64_t*)src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        a = __builtin_bit_cast(float, (uint32_t)v);
        b = __builtin_bit_cast(float, (uint32_t)(v >> 32));
      };
      auto put1 = [](float* dst, float a) {
        __hip_atomic_store((uint32_t*)dst, __builtin_bit_cast(uint32_t, a), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      };
      auto get1 = [](const float* src) -> float {
        return __builtin_bit_cast(float, __hip_atomic_load((const uint32_t*)src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      };
      // slot layout: accumulator pair (m, i/2) of wave and lane at ((m*8 + i/2)*NCOMP + wave)*128 + lane*2; then
      // three statistics per lane
      if (computes) {
        float* slot = p.sk_slots + (int64_t)(sk.slot0 + sk.kp) * SLOT_FLOATS;
#pragma unroll
        for (int m = 0; m < MTD; m++)
#pragma unroll
          for (int a = 0; a < 8; a++) put2(slot + ((m * 8 + a) * NCOMP + wave) * 128 + lane * 2, oacc[m][2 * a], oacc[m][2 * a + 1]);
        float* st = slot + D * 32 * NCOMP + wave * 64 + lane;
        put1(st, m_ref);
        put1(st + 64 * NCOMP, lsum[0] + lsum[1]);
        put1(st + 128 * NCOMP, m_true);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // compiler ordering only
      wait_fills<0>();                                           // this wave's stores have been written through
      __syncthreads();
      volatile int* flag = (volatile int*)smem;   // the K/V buffers are idle from here on
      if (tid == 0) {
        const int n = u1 - u0;
        const int old = __hip_atomic_fetch_add(p.sk_counters + w, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        flag[0] = (old + n == sk.tile_units) ? 1 : 0;
      }
      __syncthreads();
      const bool finisher = flag[0] != 0;
      __syncthreads();   // everyone has read the flag before the epilogue reuses the buffer
      if (!finisher) return;
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");   // compiler ordering only
      if (tid == 0) __hip_atomic_store(p.sk_counters + w, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // ready for the next launch
      if (computes) {
        // pass 1: common reference maximum (independent loads, one round trip); pass 2: the pieces in list order,
        // this workgroup's own included, every one read back from its slot: the same arithmetic whoever finishes
        const float* st0 = p.sk_slots + (int64_t)sk.slot0 * SLOT_FLOATS + D * 32 * NCOMP + wave * 64 + lane;
        float m_star = NEG_BIG;
        m_true = -INFINITY;
#pragma unroll
        for (int kp = 0; kp < SK_MAX_PIECES; kp++)
          if (kp < sk.pieces) {
            m_star = fmaxf(m_star, get1(st0 + (int64_t)kp * SLOT_FLOATS));
            m_true = fmaxf(m_true, get1(st0 + (int64_t)kp * SLOT_FLOATS + 128 * NCOMP));
          }
#pragma unroll
        for (int m = 0; m < MTD; m++)
#pragma unroll
          for (int i = 0; i < 16; i++) oacc[m][i] = 0.f;
        lsum[0] = lsum[1] = 0.f;
        for (int kp = 0; kp < sk.pieces; kp++) {
          const float* slot = p.sk_slots + (int64_t)(sk.slot0 + kp) * SLOT_FLOATS;
          const float* st = slot + D * 32 * NCOMP + wave * 64 + lane;
          const float alpha = fast_exp2(get1(st) - m_star);
          lsum[0] = fmaf(get1(st + 64 * NCOMP), alpha, lsum[0]);
#pragma unroll
          for (int m = 0; m < MTD; m++)
#pragma unroll
            for (int a = 0; a < 8; a++) {
              float x, y;
              get2(slot + ((m * 8 + a) * NCOMP + wave) * 128 + lane * 2, x, y);
              oacc[m][2 * a] = fmaf(x, alpha, oacc[m][2 * a]);
              oacc[m][2 * a + 1] = fmaf(y, alpha, oacc[m][2 * a + 1]);
            }
        }
        m_ref = m_star;
      }
    }
  }

  // ---- epilogue ----
  if (NPROD && wave >= NCOMP) return;   // fetch waves own no query rows (only reached with an empty list)
  const float ltot = xhalf_sum(lsum[0] + lsum[1]);
  const bool empty = !(ltot > 0.f);
  const float inv = empty ? 0.f : 1.0f / ltot;
  const int qrow_w = q0 + rblk * 32 + r;
  if (hh == 0 && half == 0 && qrow_w < p.Lq) {
    const int64_t off = ((int64_t)b * p.H + h) * p.Lq + qrow_w;
    if (p.M) p.M[off] = empty ? -INFINITY : m_true;
    if (p.L) p.L[off] = empty ? 1.0f : ltot * fast_exp2(m_ref - m_true);
    if (p.LSE2) p.LSE2[off] = empty ? -INFINITY : m_ref + __builtin_amdgcn_logf(ltot);
    if (p.RCP) p.RCP[off] = empty ? INFINITY : fast_exp2(-m_ref) * inv;
  }
  if (LSE_ONLY) return;

  const float osc = ACCUM ? p.o_scale * inv : inv;
  if constexpr (ACCUM) {
    if (p.o_accum) {
      // o = o_accum (or its bilinear upsample) + o_scale * O / l, formed in fp32 and rounded once.  The accumulators
      // go through LDS as fp32, half of the head dimension at a time (the K/V buffers hold 32 rows x D/2 floats per
      // wave), so that a lane ends up with 8 consecutive columns of one row: the o_accum rows (four taps of the
      // coarser grid when upsampling: half-pixel centres, edge clamp, src = max(0, (dst + 0.5) * src_side / dst_side
      // - 0.5), the align_corners = False rule) are then read with 16-byte loads that 8 neighbouring lanes share a
      // row of, and o is stored the same way.
      constexpr int HD = D / 2, FSTR = HD * 4 + 16, CPRH = HD / 8, ITER = (32 * CPRH) / 64;
      static_assert(NCOMP * 32 * FSTR <= 4 * TILE, "fp32 epilogue buffer must fit in the K/V buffers");
      char* fb = smem + wave * (32 * FSTR);
      const bf16_t* abase = p.o_accum + b * p.oa_sb + h * p.oa_sh;
      bf16_t* op = p.o + b * p.o_sb + h * p.o_sh;
#pragma unroll
      for (int pass = 0; pass < (PAIR ? 1 : 2); pass++) {   // (a wave of a pair holds its half alone)
#pragma unroll
        for (int mm = 0; mm < MTD / 2; mm++) {
          const int m = pass * (MTD / 2) + mm;
#pragma unroll
          for (int a = 0; a < 4; a++) {
            const f32x4 x = {oacc[m][4 * a + 0] * osc, oacc[m][4 * a + 1] * osc, oacc[m][4 * a + 2] * osc, oacc[m][4 * a + 3] * osc};
            *(f32x4*)(fb + r * FSTR + (mm * 32 + 8 * a + 4 * hh) * 4) = x;
          }
        }
        // each wave re-reads only its own 32 rows: a wave-local fence is enough
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < ITER; i++) {
          const int cidx = lane + i * 64;
          const int orow = cidx / CPRH, oc = cidx - orow * CPRH;
          const int grow = q0 + rblk * 32 + orow;
          if (grow < p.Lq) {
            const f32x4 xa = *(const f32x4*)(fb + orow * FSTR + oc * 32), xb = *(const f32x4*)(fb + orow * FSTR + oc * 32 + 16);
            float x[8] = {xa[0], xa[1], xa[2], xa[3], xb[0], xb[1], xb[2], xb[3]};
            const int col = (PAIR ? half : pass) * HD + oc * 8;
            if (p.up_src > 0) {
              const int y = grow / p.up_dst, xq = grow - y * p.up_dst;
              const float sc = (float)p.up_src / (float)p.up_dst;
              const float sy = fmaxf(sc * ((float)y + 0.5f) - 0.5f, 0.f), sx = fmaxf(sc * ((float)xq + 0.5f) - 0.5f, 0.f);
              const int y0 = min((int)sy, p.up_src - 1), x0 = min((int)sx, p.up_src - 1);
              const int y1 = min(y0 + 1, p.up_src - 1), x1 = min(x0 + 1, p.up_src - 1);
              const float wy1 = sy - (float)y0, wx1 = sx - (float)x0, wy0 = 1.f - wy1, wx0 = 1.f - wx1;
              const u32x4 t00 = *(const u32x4*)(abase + (int64_t)(y0 * p.up_src + x0) * p.oa_sr + col);
              const u32x4 t01 = *(const u32x4*)(abase + (int64_t)(y0 * p.up_src + x1) * p.oa_sr + col);
              const u32x4 t10 = *(const u32x4*)(abase + (int64_t)(y1 * p.up_src + x0) * p.oa_sr + col);
              const u32x4 t11 = *(const u32x4*)(abase + (int64_t)(y1 * p.up_src + x1) * p.oa_sr + col);
#pragma unroll
              for (int e = 0; e < 4; e++) {
                x[2 * e] += wy0 * (wx0 * bf16_lo(t00[e]) + wx1 * bf16_lo(t01[e])) + wy1 * (wx0 * bf16_lo(t10[e]) + wx1 * bf16_lo(t11[e]));
                x[2 * e + 1] += wy0 * (wx0 * bf16_hi(t00[e]) + wx1 * bf16_hi(t01[e])) + wy1 * (wx0 * bf16_hi(t10[e]) + wx1 * bf16_hi(t11[e]));
              }
            } else {
              const u32x4 t = *(const u32x4*)(abase + (int64_t)grow * p.oa_sr + col);
#pragma unroll
              for (int e = 0; e < 4; e++) { x[2 * e] += bf16_lo(t[e]); x[2 * e + 1] += bf16_hi(t[e]); }
            }
            const u32x4 val = {pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3]), pack_bf16(x[4], x[5]), pack_bf16(x[6], x[7])};
            *(u32x4*)(op + (int64_t)grow * p.o_sr + col) = val;
          }
        }
        __builtin_amdgcn_wave_barrier();   // the buffer is rewritten by the next pass
      }
      return;
    }
  }
  char* ob = smem + rblk * (32 * OSTR) + half * D;   // a pair: each wave its columns
#pragma unroll
  for (int m = 0; m < MTW; m++) {
#pragma unroll
    for (int a = 0; a < 4; a++) {
      const int dcol = m * 32 + 8 * a + 4 * hh;
      float x0 = oacc[m][4 * a + 0] * osc, x1 = oacc[m][4 * a + 1] * osc;
      float x2 = oacc[m][4 * a + 2] * osc, x3 = oacc[m][4 * a + 3] * osc;
      u32x2 pk = {pack_bf16(x0, x1), pack_bf16(x2, x3)};
      *(u32x2*)(ob + r * OSTR + dcol * 2) = pk;
    }
  }
  // each wave re-reads only its own 32 rows: a wave-local fence is enough
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_wave_barrier();
  bf16_t* op = p.o + b * p.o_sb + h * p.o_sh;
  constexpr int OCPR = MTW * 4;
#pragma unroll
  for (int i = 0; i < (32 * OCPR) / 64; i++) {
    const int cidx = lane + i * 64;
    const int orow = cidx / OCPR, ocol = cidx - orow * OCPR;
    const int grow = q0 + rblk * 32 + orow;
    if (grow < p.Lq) {
      u32x4 val = *(const u32x4*)(ob + orow * OSTR + ocol * 16);
      *(u32x4*)(op + (int64_t)grow * p.o_sr + half * (D / 2) + ocol * 8) = val;
    }
  }
}
#endif  // __HIP_DEVICE_COMPILE__

// The tile of slice bh with its place-th longest list, of the n tiles that run in order (see ranked_slice)
template <int WGROWS>
__device__ __forceinline__ int tile_by_length(const AttnParams& p, int bh, int place, int n) {
  const int lane = __builtin_amdgcn_workitem_id_x() & 63, b = bh / p.H, h = bh - b * p.H;
  const int g = lane * WGROWS / p.group_rows;
  const int raw = lane < n ? p.cnt[b * p.cnt_sb + h * p.cnt_sh + g] : 0;
  // the heads of all lists are asked for at the same time: whichever is read next is then in the L2
  const int head = lane < n && p.list_len > 0 ? p.list[b * p.list_sb + h * p.list_sh + (int64_t)g * p.list_sg] : 0;
  asm volatile("" : : "v"(head), "v"(raw));
  const int len = max(0, min(raw, p.list_len));
  if (__builtin_amdgcn_ballot_w64(lane < n && len != __builtin_amdgcn_readfirstlane(len)) == 0) return place;
  const int key = lane < n ? (len << 6) + 63 - lane : -1;   // length and position in one number; never equal
  int longer = 0;
  for (int k = 0; k < n; k++) longer += __builtin_amdgcn_readlane(key, k) > key ? 1 : 0;
  return __builtin_ctzll(__builtin_amdgcn_ballot_w64(lane < n && longer == place));
}

template <int D, int NWAVES, int MODE, bool LSE_ONLY>
constexpr bool ranks_tiles = MODE == MODE_BLOCK && !LSE_ONLY && D == 128 && NWAVES == 4;

// THIRD: registers of a wave limited so that three workgroups share a compute unit, see third_workgroup
template <int D, int NWAVES, int MODE, bool ACCUM, bool LSE_ONLY, int NPROD, bool IDLE, bool THIRD = false, bool PAIR = false>
__global__ __launch_bounds__(NWAVES * 64, ((NWAVES <= 4 && D <= 128) ? (THIRD ? 3 : 2) : 1)) void attn_fwd_kernel(const AttnParams p) {
  // The body is compiled for the device only: the host pass just needs the launch stub, and it
  // silently drops the stub when the body uses the LDS-DMA builtins.
#if defined(__HIP_DEVICE_COMPILE__)
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  // The place is worked out in scalar registers (blockIdx would be a call, as threadIdx: library functions are compiled with the
  // target's own features and so not inlined here, and their result counts as different per lane) and then handed on as if it
  // differed per lane: known to be uniform, it leads the compiler to 30 .. 40 more vector registers, and spills.
  // One field of every 64-byte line of the arguments is asked for ahead of that, so that their first reads are one round trip
  // to memory, not one for the order, one for the shape and one for the pointers behind each other (1 x 3, d256 6.98 -> 6.83 us;
  // sparse step 30 x 30 d64 20.7 -> 20.3).
  asm volatile("" : : "s"(p.q), "s"(p.q_sb), "s"(p.v_sb), "s"(p.o_sh), "s"(p.H), "s"(p.list_sb));
  int bh, qt;
  if (!tile_of(p.order, __builtin_amdgcn_workgroup_id_x(), bh, qt)) return;
  if constexpr (ranks_tiles<D, NWAVES, MODE, LSE_ONLY>) {
    const int x = __builtin_amdgcn_workgroup_id_x() % TILE_XCDS;
    if (p.last_round > 0 && qt < p.order.nqt && ranked_slice(p.order, bh, x, p.last_round)) qt = tile_by_length<NWAVES * 32>(p, bh, qt, p.order.nqt);
  }
  asm volatile("" : "+v"(bh), "+v"(qt));
  attn_item<D, NWAVES, MODE, ACCUM, LSE_ONLY, false, NPROD, IDLE, PAIR, THIRD>(p, smem, 0, bh, qt, 0, 0, true, SkCtx{});
#endif
}

// Balanced launch: every workgroup runs one item of the partition described in sk_partition.h, which it reads from
// the item table built by plan_kernel, or, for dense attention (all lists equally long, sk_uniform_n pieces per
// tile), computes from its index.
template <int D, int NWAVES, int MODE, bool ACCUM>
__global__ __launch_bounds__(NWAVES * 64, (NWAVES <= 4 ? 2 : 1)) void attn_fwd_balanced_kernel(const AttnParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int N = p.total_wg;
  const bool uniform = p.sk_uniform_n > 0;
  const int items = uniform ? N * p.sk_uniform_n : min(max(p.sk_plan[1], 0), (int)gridDim.x);
  // consecutive items go to the same XCD (workgroup ids are dealt round-robin to the 8 XCDs): the K/V of a head
  // stay in its L2 and the pieces of a query tile meet there
  const int per_xcd = (items + 7) >> 3;
  const int slot_in_xcd = blockIdx.x >> 3;
  const int k = (blockIdx.x & 7) * per_xcd + slot_in_xcd;
  if (slot_in_xcd >= per_xcd || k >= items) return;
  SkCtx sk;
  int w, u0, u1;
  if (uniform) {
    const int n = p.sk_uniform_n, T = (p.Lk + 63) >> 6;
    w = k / n;
    sk.kp = k - w * n;
    sk.pieces = n;
    sk.slot0 = w * n;
    sk.tile_units = T;
    sk_piece(T, n, sk.kp, u0, u1);
  } else {
    const int* it = p.sk_plan + SK_PLAN_HEADER + SK_PLAN_ITEM * k;
    w = max(0, min(it[0], N - 1));
    u0 = it[1];
    u1 = it[2];
    sk.slot0 = it[3];
    sk.pieces = it[4];
    sk.kp = it[5];
    sk.tile_units = it[6];
    // a damaged table must not send a store outside the workspace
    if (sk.pieces < 1 || sk.pieces > SK_MAX_PIECES || sk.kp < 0 || sk.kp >= sk.pieces || (sk.pieces > 1 && (sk.slot0 < 0 || sk.slot0 + sk.pieces > 2 * p.sk_wgs))) return;
  }
  const int bh = w / p.nqt;
  attn_item<D, NWAVES, MODE, ACCUM, false, true, (MODE == MODE_GATHER && NWAVES == 8) ? 2 : 0, false>(p, smem, w, bh, w - bh * p.nqt, u0, u1, sk.pieces == 1, sk);
#endif
}

// words [0, n) of a device buffer := 0 (a kernel, not hipMemsetAsync: callers may be capturing a HIP graph)
__global__ void zero_words_kernel(uint32_t* dst, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = 0u;
}

// Item table of a balanced launch over tile lists, from the list lengths: one workgroup.  Also clears the arrival
// counters of the launch's query tiles, so that a launch does not depend on what the last one left in the workspace.
template <int WGROWS, int MODE>
__global__ __launch_bounds__(256) void plan_kernel(const AttnParams p, int* plan) {
  __shared__ int units[SK_MAX_QTILES];    // units of tile u
  __shared__ int ipfx[SK_MAX_QTILES + 1]; // items before tile u
  __shared__ int spfx[SK_MAX_QTILES + 1]; // slots before tile u
  __shared__ int total[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int N = p.total_wg;
  for (int u = tid; u < N; u += 256) {
    const int bh = u / p.nqt, qt = u - bh * p.nqt;
    const int b = bh / p.H, h = bh - b * p.H;
    const int g = (qt * WGROWS) / p.group_rows;
    const int cnt = max(0, min(p.cnt[b * p.cnt_sb + h * p.cnt_sh + g], p.list_len));
    units[u] = (MODE == MODE_BLOCK) ? cnt : ((cnt + 63) >> 6);
    p.sk_counters[u] = 0;
  }
  __syncthreads();
  if (wave == 0) {
    // every lane owns a run of consecutive tiles; U first, then the two prefix tables
    const int per = (N + 63) >> 6, first = lane * per;
    int sum = 0;
    for (int j = 0; j < per; j++)
      if (first + j < N) sum += max(units[first + j], 1);
    int U = sum;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) U += __shfl_xor(U, d, 64);
    int S = sk_share(U, p.sk_wgs, p.sk_min_share);
    const bool cut = sk_worth_cutting(U, S, N, p.sk_wgs);
    int it = 0, sl = 0;
    for (int j = 0; j < per; j++)
      if (first + j < N) {
        const int n = cut ? sk_pieces(units[first + j], S, p.sk_min_piece) : 1;
        it += n;
        sl += n > 1 ? n : 0;
      }
    int it_incl = it, sl_incl = sl;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int a = __shfl_up(it_incl, d, 64), c = __shfl_up(sl_incl, d, 64);
      if (lane >= d) { it_incl += a; sl_incl += c; }
    }
    int irun = it_incl - it, srun = sl_incl - sl;
    for (int j = 0; j < per; j++)
      if (first + j < N) {
        const int n = cut ? sk_pieces(units[first + j], S, p.sk_min_piece) : 1;
        ipfx[first + j] = irun;
        spfx[first + j] = srun;
        irun += n;
        srun += n > 1 ? n : 0;
      }
    if (lane == 63) { total[0] = it_incl; total[1] = sl_incl; total[2] = S; total[3] = cut ? 1 : 0; }
  }
  __syncthreads();
  const int S = total[2];
  const bool cut = total[3] != 0;
  // the pieces-per-share bound keeps both totals inside the launch (N + sk_wgs items) and the workspace (2 * sk_wgs
  // slots); if a list-length table breaks it after all, every tile stays whole
  const bool fits = total[0] <= N + p.sk_wgs && total[1] <= 2 * p.sk_wgs;
  if (tid == 0) {
    plan[0] = SK_PLAN_MAGIC;
    plan[1] = fits ? total[0] : N;
    plan[2] = N;
    plan[3] = S;
    plan[4] = fits ? total[1] : 0;
    plan[5] = plan[6] = plan[7] = 0;
  }
  for (int u = tid; u < N; u += 256) {
    const int T = units[u];
    const int n = (cut && fits) ? sk_pieces(T, S, p.sk_min_piece) : 1;
    const int base = fits ? ipfx[u] : u;
    for (int kp = 0; kp < n; kp++) {
      int u0, u1;
      sk_piece(T, n, kp, u0, u1);
      int* it = plan + SK_PLAN_HEADER + SK_PLAN_ITEM * (base + kp);
      it[0] = u; it[1] = u0; it[2] = u1; it[3] = n > 1 ? spfx[u] : -1;
      it[4] = n; it[5] = kp; it[6] = T; it[7] = 0;
    }
  }
}

// Three 128-row workgroups per compute unit at head_dim 64: 168 registers per wave instead of 174, two of them spilled.  Where
// two per compute unit hold the launch the third slot stays empty and the spills cost 1 to 2 % (two against three, lists of 30 %:
// B2 H12 1600 x 4121 30.8 / 31.4 us, B2 H16 2048 x 4121 35.0 / 35.3); larger launches are up to 10 % faster (B3 H24 1024 x 1100
// 37.1 / 33.4 us, B2 H17 2048 x 4121 117 / 107, B2 H16 2304 x 6425 179 / 165, in lists of 25 % 49.4 / 45.6).  The 2-wave workgroups of
// 64-row query blocks are not (B2 H16 4096 x 10521 in lists of 30 %: 149 / 162 us).
static bool third_workgroup(int total_wg) { return total_wg > 2 * device_cus(); }

// Lists whose lengths a wave can rank, one tile per lane.
static bool lists_by_length(const AttnParams& p) { return p.list && p.order.nqt > 1 && p.order.nqt <= 64; }

template <int D, int NWAVES, int MODE, bool ACCUM, bool LSE_ONLY, int NPROD = (MODE == MODE_GATHER && NWAVES == 8) ? 2 : 0, bool PAIR = false>
static int launch_one(const AttnParams& p0, hipStream_t stream) {
  AttnParams p = p0;
  if (p.kv_group < 1) p.kv_group = 1;
  constexpr int WGROWS = (NWAVES - NPROD) * (PAIR ? 16 : 32);
  constexpr int SMEM = attn_lds_bytes<D, NWAVES - NPROD, MODE, PAIR>();
  if (MODE == MODE_BLOCK && p.list == nullptr) p.group_rows = WGROWS;  // dense: any row grouping
  if (p.group_rows % WGROWS != 0) return LVAR_EINVAL;
  if (p.remap_gs > 0 && !reads_remapped<D, NWAVES, MODE, NPROD>) return LVAR_EUNSUPPORTED;
  p.nqt = (p.Lq + WGROWS - 1) / WGROWS;
  p.total_wg = p.B * p.H * p.nqt;
  constexpr bool WIDE = MODE == MODE_BLOCK && NWAVES == 8;   // 256 query rows, or 128 and fetch waves
  if constexpr (!LSE_ONLY && NPROD != 4) {
    const bool dense = (MODE == MODE_BLOCK && p.list == nullptr);
    const int64_t per_tile = (MODE == MODE_BLOCK) ? (p.list ? p.list_len : (p.Lk + 63) / 64) : (p.list_len + 63) / 64;
    const int sub = (MODE == MODE_BLOCK && p.list) ? p.sub_shift : 0;
    // (64-row query blocks always take the plain launch)
    p.sk_wgs = (p.sk_ws && NWAVES != 2 && !WIDE && D <= 128) ? sk_plan(p.total_wg, NWAVES, sk_slot_floats(D, MODE, NWAVES), per_tile, sub, p.sk_ws_bytes,
                                 p.sk_min_share, p.sk_min_piece) : 0;
    p.sk_uniform_n = 0;
    if (p.sk_wgs > 0 && dense) {
      // all lists have (Lk + 63) / 64 entries: the pieces per tile follow from the sizes alone
      p.sk_uniform_n = sk_dense_pieces(p.total_wg, (int)per_tile, p.sk_wgs, p.sk_min_share, p.sk_min_piece);
      if (p.sk_uniform_n == 0) p.sk_wgs = 0;   // whole tiles: the plain launch
    }
    if constexpr (NWAVES != 2 && !WIDE && D <= 128) if (p.sk_wgs > 0) {
      p.sk_counters = (int*)p.sk_ws;
      p.sk_slots = (float*)((char*)p.sk_ws + SK_COUNTER_BYTES + sk_plan_bytes(p.sk_wgs));
      int grid_sk;
      if (p.sk_uniform_n > 0 || p.sk_plan) {
        // no table kernel ahead of this launch: the arrival counters are cleared by a fill of their own
        hipLaunchKernelGGL(zero_words_kernel, dim3((p.total_wg + 255) / 256), dim3(256), 0, stream, (uint32_t*)p.sk_counters, p.total_wg);
        if (hipGetLastError() != hipSuccess) return LVAR_ELAUNCH;
      }
      if (p.sk_uniform_n > 0) {
        grid_sk = ((p.total_wg * p.sk_uniform_n + 7) / 8) * 8;
      } else {
        if (!p.sk_plan) {
          // no table from the caller: build it now, in the workspace
          int* plan = (int*)((char*)p.sk_ws + SK_COUNTER_BYTES);
          hipLaunchKernelGGL((plan_kernel<WGROWS, MODE>), dim3(1), dim3(256), 0, stream, p, plan);
          if (hipGetLastError() != hipSuccess) return LVAR_ELAUNCH;
          p.sk_plan = plan;
        }
        grid_sk = ((p.total_wg + p.sk_wgs + 7) / 8) * 8;   // at most one item per query tile plus one per share
      }
      auto kern = attn_fwd_balanced_kernel<D, NWAVES, MODE, ACCUM>;
      static std::atomic<uint64_t> lds_ready_sk{0};
      if (!ensure_lds_limit((const void*)kern, SMEM, lds_ready_sk)) return LVAR_ELAUNCH;
      hipLaunchKernelGGL(kern, dim3(grid_sk), dim3(NWAVES * 64), SMEM, stream, p);
      return hipGetLastError() == hipSuccess ? LVAR_OK : LVAR_ELAUNCH;
    }
  }
  if constexpr (MODE == MODE_BLOCK && !LSE_ONLY && NWAVES == 4) {
    const BlockForm form = block_form((int64_t)p.B * p.H, p.Lq, p.Lk, D, p.list != nullptr, p.group_rows, device_cus());
    if (form == BlockForm::PAIRS) return launch_one<D, 8, MODE_BLOCK, false, false, 4, true>(p0, stream);
    if constexpr (D <= 128) {
      if (form == BlockForm::WIDE) return launch_one<D, 8, MODE_BLOCK, false, false>(p0, stream);
      if (form == BlockForm::ROWS_96) return launch_one<D, 7, MODE_BLOCK, false, false, 4>(p0, stream);
      if (form == BlockForm::FETCH) return launch_one<D, 8, MODE_BLOCK, false, false, 4>(p0, stream);
    }
  }
  const int rest = p.Lq % WGROWS;
  const bool ragged = MODE == MODE_GATHER ? NPROD > 0 && ragged_runs_last(p.B * p.H, p.nqt, rest, WGROWS, device_cus())
                                          : p.list != nullptr && ragged_lists_last(p.B * p.H, p.nqt, rest, device_cus());
  p.order = tile_order(p.B * p.H, p.nqt, ragged);
  const int grid = TILE_XCDS * p.order.per_xcd;
  if constexpr (ranks_tiles<D, NWAVES, MODE, LSE_ONLY>) p.last_round = lists_by_length(p) ? short_last_round(p.order, device_cus() / TILE_XCDS * 2) : 0;
  if constexpr (D == 64 && NWAVES == 4 && MODE == MODE_BLOCK && !LSE_ONLY) {
    if (third_workgroup(p.total_wg)) {
      static_assert(SMEM <= 48 * 1024, "three workgroups share the LDS of a compute unit; no larger limit has to be asked for");
      hipLaunchKernelGGL((attn_fwd_kernel<D, NWAVES, MODE, ACCUM, LSE_ONLY, NPROD, false, true>), dim3(grid), dim3(NWAVES * 64), SMEM, stream, p);
      return hipGetLastError() == hipSuccess ? LVAR_OK : LVAR_ELAUNCH;
    }
  }
  // (an instance of its own; not at head_dim 64, where the role's registers have to be spilled, nor at 256: +1 % with it)
  if constexpr (MODE == MODE_BLOCK && D == 128 && NPROD == 0 && NWAVES >= 4) {
    if (idle_waves_pay(NWAVES, p.nqt, rest)) {
      auto kern = attn_fwd_kernel<D, NWAVES, MODE, ACCUM, LSE_ONLY, NPROD, true>;
      static std::atomic<uint64_t> lds_ready{0};
      if (!ensure_lds_limit((const void*)kern, SMEM, lds_ready)) return LVAR_ELAUNCH;
      hipLaunchKernelGGL(kern, dim3(grid), dim3(NWAVES * 64), SMEM, stream, p);
      return hipGetLastError() == hipSuccess ? LVAR_OK : LVAR_ELAUNCH;
    }
  }
  auto kern = attn_fwd_kernel<D, NWAVES, MODE, ACCUM, LSE_ONLY, NPROD, false, false, PAIR>;
  static std::atomic<uint64_t> lds_ready{0};
  if (!ensure_lds_limit((const void*)kern, SMEM, lds_ready)) return LVAR_ELAUNCH;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(NWAVES * 64), SMEM, stream, p);
  return hipGetLastError() == hipSuccess ? LVAR_OK : LVAR_ELAUNCH;
}

template <int D>
static int launch_d(const AttnParams& p, int mode, bool accum, bool lse_only, int nwaves, hipStream_t s) {
  if (mode == MODE_BLOCK) {
    if (nwaves == 2 && !lse_only) return launch_one<D, 2, MODE_BLOCK, false, false>(p, s);   // 64-row query blocks
    if (nwaves != 4) return LVAR_EUNSUPPORTED;
    return lse_only ? launch_one<D, 4, MODE_BLOCK, false, true>(p, s) : launch_one<D, 4, MODE_BLOCK, false, false>(p, s);
  } else if (mode == MODE_GATHER) {
    // (head_dim 256: a wave needs more than 256 registers, so one wave per SIMD: 192-row groups run as two 3-wave workgroups)
    if constexpr (D > 128) {
      if (nwaves == 8) nwaves = 3;
    } else if (nwaves == 8) {
      const TokenForm form = p.sk_ws ? TokenForm::PLAIN : token_form((int64_t)p.B * p.H, p.Lq, D, device_cus());
      if (form == TokenForm::PAIRS) return launch_one<D, 8, MODE_GATHER, true, false, 4, true>(p, s);
      if (form == TokenForm::HALF_GROUPS) return launch_one<D, 7, MODE_GATHER, true, false, 4>(p, s);
      if constexpr (D == 64) if (form == TokenForm::THREE_WAVES) return launch_one<D, 3, MODE_GATHER, true, false>(p, s);
      return launch_one<D, 8, MODE_GATHER, true, false>(p, s);
    }
    if (nwaves == 3) return launch_one<D, 3, MODE_GATHER, true, false>(p, s);
    if (nwaves == 2) return launch_one<D, 2, MODE_GATHER, true, false>(p, s);
  }
  return LVAR_EUNSUPPORTED;
}

int launch_attn(const AttnParams& p, int head_dim, int mode, bool accum, bool lse_only, int nwaves, hipStream_t s) {
  if (head_dim == 128) return launch_d<128>(p, mode, accum, lse_only, nwaves, s);
  if (head_dim == 64) return launch_d<64>(p, mode, accum, lse_only, nwaves, s);
  if (head_dim == 256) return launch_d<256>(p, mode, accum, lse_only, nwaves, s);
  return LVAR_EUNSUPPORTED;
}

int device_cus() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  const int slot = dev & 63;
  int n = cached[slot].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 0;
    cached[slot].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Workgroups of the balanced launch, or 0 for the plain launch.  Balanced when the plain grid would leave the chip
// unevenly filled, i.e. fewer than four rounds of workgroups: one workgroup per resident slot (two per CU for the
// 4-wave kernels), or one per CU if the workspace only holds that many slot pairs.  `per_tile` is an upper bound
// of the list entries of a query tile; min_share / min_piece come in as 64-key tiles (0 = default) and go out
// as list entries (a list entry of a 128-key block list is two tiles: sub = 1).
int sk_plan(int total_wg, int nwaves, int slot_floats, int64_t per_tile, int sub, int64_t ws_bytes, int& min_share, int& min_piece) {
  const int cus = device_cus();
  const int slots = cus * (nwaves <= 4 ? 2 : 1);
  if (cus < 8 || cus % 8 != 0 || total_wg > SK_MAX_QTILES || total_wg >= 4 * slots || ws_bytes <= SK_COUNTER_BYTES) return 0;
  if (per_tile * total_wg >= (1ll << 30)) return 0;   // unit counts stay well inside 32 bits
  auto fits = [&](int P) { return SK_COUNTER_BYTES + sk_plan_bytes(P) + 2 * (int64_t)P * slot_floats * 4 <= ws_bytes; };
  const int P = fits(slots) ? slots : (fits(cus) ? cus : 0);
  const int share = min_share > 0 ? min_share : 8, piece = min_piece > 0 ? min_piece : 4;
  min_piece = (piece >> sub) > 0 ? (piece >> sub) : 1;
  min_share = (share >> sub) > min_piece ? (share >> sub) : min_piece;   // shares no smaller than pieces
  // With fewer query tiles than slots the plain launch already runs them all at once, and cutting only pays if
  // it makes the longest walk shorter: lists of at least one and a half shares (were every list full; the kernel
  // looks at the real lists and leaves the tiles whole if they are shorter).
  if (P == 0) return 0;
  if (total_wg < slots && 2 * per_tile < 3 * (int64_t)min_share) return 0;
  return P;
}

// Pieces per query tile of a balanced dense launch (every list has T tiles) on sk_wgs shares, or 0 when the tiles
// stay whole or the pieces would not fit the launch's slots: then the launch is the plain one.
int sk_dense_pieces(int total_wg, int T, int sk_wgs, int min_share, int min_piece) {
  if (sk_wgs <= 0 || total_wg <= 0 || T <= 0) return 0;
  const int U = total_wg * T;
  const int S = sk_share(U, sk_wgs, min_share);
  const int n = sk_worth_cutting(U, S, total_wg, sk_wgs) ? sk_pieces(T, S, min_piece) : 1;
  return (n > 1 && (int64_t)n * total_wg <= 2 * (int64_t)sk_wgs) ? n : 0;
}

// bytes of the item-table area of a workspace for P shares (256-byte granules)
int64_t sk_plan_bytes(int P) {
  const int64_t b = (int64_t)(SK_PLAN_HEADER + SK_PLAN_ITEM * (SK_MAX_QTILES + P)) * 4;
  return (b + 255) / 256 * 256;
}

// floats of one workspace slot of a balanced launch: the accumulators and three statistics of every lane
int sk_slot_floats(int head_dim, int mode, int nwaves) {
  const int ncomp = (mode == MODE_GATHER && nwaves == 8) ? 6 : nwaves;
  return head_dim * 32 * ncomp + 3 * 64 * ncomp;
}

}  // namespace lvar
