// Persistent ping-pong block-scaled GEMM for large problems (gfx950): 256 x 256 tile, 8 waves.
//
// Same math, operand layouts and LDS swizzle as the kernel in mx_gemm_mfma.hip; what differs is the
// schedule.  The 8 waves form two teams of four (one wave of each team per SIMD): team 0 owns rows
// 0-127 of the tile, team 1 rows 128-255; wave (team, wn) computes the 128 x 64 block at columns
// 64 wn.  Every K stage of a wave is split into
//   a MEMORY phase: LDS-DMA issue for stage s + 2, LDS reads of the B fragments and the first A
//                   tiles of stage s;
//   an MFMA phase:  32 (64 for FP4) back-to-back MFMAs from registers, with the reads of the other
//                   remaining A tiles slotted in 8 or 16 MFMAs ahead of their use.
// One s_barrier ends every phase.  Team 1 runs exactly one phase behind team 0 (it executes one extra
// barrier before its first stage, team 0 one extra after its last), so the two waves of a SIMD are
// never in the same phase: while one waits on LDS, issues DMA or sits in a barrier, the other feeds
// the matrix pipe.
//
// LDS: three A stage buffers (stage s lives in buffer s % 3) and two B stage buffers (s % 2), exactly
// 160 KiB for 128-byte stage rows.  A DMA load is issued two stages ahead of its use.
//   A rows: wave (T, wn) loads a quarter of team T's 128 rows; only team T reads them.
//   B rows: wave (1, wn) loads all 64 rows of column block wn (the rows only waves (0, wn) and (1, wn)
//           read) for stage s + 2 into the buffer of stage s, right after its own reads of stage s;
//           wave (0, wn) read them one phase earlier and will read the new contents three phases
//           later, behind the barrier at which team 1 waits for the loads (vmcnt).
//
// Persistence: a workgroup walks a list of tiles.  The stage pipeline runs straight across tile
// boundaries (the last two stages of a tile prefetch the first two of the next one), and the output
// of a finished tile is converted and stored inside the first memory phase of the next tile, i.e.
// while the other team is in an MFMA phase, so neither the pipeline fill nor the epilogue idles the
// matrix pipe.  A workgroup is given more than one tile only when a tile has at least two stages and
// a whole number of K-quads (K a multiple of 512).
//
// Last round: tiles that would leave most of the workgroups idle are split along K among them (SPLIT; tail_splits in
// mx_gemm_pp.h says when), each workgroup's last tile then being some K-quads of one.  The sums leave as they lie in the
// registers (1 KiB per store) and pp_tail_kernel adds and writes them.  The grouped form knows how many slots hold rows
// only on the device (num_slots) and walks the tiles of those.  4096 tokens x 2 in 8 experts, 4096 x 14336 MXFP8: the first
// projection, 18 rounds of the upper bound's 39 tile rows, 929 -> 868 us; the second, 2.25 rounds, 514 -> 413 + 17 us.
#include <stdlib.h>

#include <type_traits>

#include "mx_gemm_pp.h"

namespace mx {
namespace {

// KTAIL: K is not a whole number of stages (or there is a single stage): the 16-byte chunks beyond the end of K are
// masked lane by lane at issue time.  Without it the loads take their precomputed offsets as they are, which keeps a
// compare and a select per DMA instruction out of the memory phase.
// SPLIT: the walk may end with a K range of one more tile, whose sums go to g.tail.  (An instance of its own: the few scalars
// more cost the whole-round products, MXFP4 8192^3 232.2 -> 234.0 us.)
template <class C, typename OutT, bool GROUPED, bool SPLIT, int TEAM, bool KTAIL>
__device__ __forceinline__ void pp_body(const GemmArgs& g, lds_u8* const smem, const int wn,
                                        const int lane, const TileWalk& walk) {
  using P = PP<C>;
  constexpr int AL = P::AL, BL = P::BL;
  // A tiles (of 8) whose fragments are read in the memory phase; the others are read inside the MFMA phase,
  // 8 MFMAs ahead of their use.  Two measured best (four: 1.5 % slower on MXFP8, 5 % on the grouped
  // variant: the longer memory phase costs more than the later reads)
  constexpr int EARLY = 2;
  constexpr int MT = C::MT;          // A tiles of a wave: 8 (6 with tiles of 192 rows)
  const int r = lane & 15, gq = lane >> 4;
  constexpr int wm0 = TEAM * C::WTM;
  constexpr int at0 = wm0 % 64 / 16; // the first one's place in its 64-row scale group
  static_assert(MT == 8 || !(GROUPED || SPLIT), "");
  const int wn0 = wn * 64;

  const int Kb_a = g.K * C::A_EB / 8, Kb_b = g.K * C::B_EB / 8;
  const int ksteps = (g.K + 127) / 128;
  const int nstages = (ksteps + C::KSUB - 1) / C::KSUB;
  const int KQ = (ksteps + 3) / 4;
  constexpr int SPQ = 4 / C::KSUB;   // stages per K-quad
  const int a_groups = (g.M + 63) / 64, b_groups = (g.N + 63) / 64;
  const __amdgpu_buffer_rsrc_t rsA = make_rsrc(g.A, operand_bytes(g.a_rows, g.lda, Kb_a));

  // ---- load context: where the DMA and scale loads of the tile being FETCHED point --------------------
  // A: instruction q of the wave covers tile rows wm0 + (4 q + wn) * A_RPI ...; B (team 1 only):
  // rows wn0 + q * B_RPI ....  A: the swizzled byte column of instruction q is col0 ^ (4 q % CPR) * 16.
  uint32_t a_voff[AL], b_voff[TEAM ? BL : 1];
  const int a_row0 = wm0 + wn * P::A_RPI + lane / C::A_CPR;
  const int a_col0 = ((lane % C::A_CPR) ^ swz<C::A_CPR>(a_row0)) * 16;
  // swizzled byte column of DMA instruction q (rows b_row0 + q * B_RPI ...)
  auto b_col = [&](int q, int lane) { return ((lane % C::B_CPR) ^ swz_bperm<C::B_CPR>(lane / C::B_CPR + q * P::B_RPI)) * 16; };
  __amdgpu_buffer_rsrc_t rsB;
  // ---- scales (native layout, mx_common.h): 16 bytes per (64-row group, K-quad, lane), dword t = K-step t of the
  // quad, byte = 16-row tile of the group (B: in the bperm_row order of the fragments).  A K-quad needs the team's
  // two A groups and the wave's one B group: three 16-byte loads (1 KiB contiguous per wave) through buffer
  // descriptors, the (group, quad) part of the address in the scalar offset.
  // as / bs _cur, _nxt: byte offset of (group, K-quad 0) for the tile being computed / being fetched.
  int as_cur[2], bs_cur, as_nxt[2], bs_nxt;
  const __amdgpu_buffer_rsrc_t rsAs = make_rsrc(g.As, (uint32_t)(packed_scale_dwords(g.M, g.K) * 4));
  const __amdgpu_buffer_rsrc_t rsBs =
      make_rsrc(g.Bs, (uint32_t)((GROUPED ? (int64_t)(g.num_experts - 1) * g.bs_expert_stride * 4 : 0) +
                                 packed_scale_dwords(g.N, g.K) * 4));
  const int sc_voff = lane * 16;
  constexpr int NSC = 3;           // scale load instructions per K-quad
  v4i sa[2], sb;
  auto load_scales = [&](const int* as_off, int bs_off, int Qn) {
#pragma unroll
    for (int u = 0; u < 2; ++u) sa[u] = __builtin_amdgcn_raw_buffer_load_b128(rsAs, sc_voff, as_off[u] + Qn * 1024, 0);
    sb = __builtin_amdgcn_raw_buffer_load_b128(rsBs, sc_voff, bs_off + Qn * 1024, 0);
  };
  bool fetch_valid = true;   // false once the walk has no further tile: loads become zero-fill no-ops
  // grouped: none of this team's 128 slots of the tile holds a routed row (every slot is looked at: two per lane,
  // then a vote, so a sentinel in front of valid ids does not hide them).  Such a half has nothing to multiply:
  // its fragment reads and MFMAs are skipped.
  bool skip_cur = false, skip_nxt = false;
  // grouped: routed-slot ids of the team's 128 rows, two per lane (lane l: rows l and 64 + l; -1 where there is no slot): of
  // the tile to be fetched next, then again of the tile being computed, whose output they place.  They and the expert are
  // requested a stage or more before the tile's first loads are set up (each DMA instruction's rows read their own ids in that
  // memory phase before, one after the other, while both teams waited).  With the walk by experts (ExpertRuns) the layer of
  // 4096 tokens, 8 experts, top 2, 4096 x 14336 takes 1400 us instead of 1445; the ids alone gave 0.5 % of it.
  int eid[2] = {-1, -1}, expert_nxt = 0;
  // grouped: origin of the tile being computed, being fetched; the columns of the one written next (the last one computed)
  int n_out = 0, m_cur = 0, n_cur = 0, m_nxt = 0, n_nxt = 0;
  ExpertRuns runs = {g.sorted_expert_ids, g.tile_m, walk.tiles_m, walk.tiles_n};
  auto load_row_ids = [&](bool valid, int m0) {
    int l = lane;
    asm volatile("" : "+v"(l));   // (nothing of this is kept in registers from one tile to the next)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int m = m0 + wm0 + 64 * u + l;
      eid[u] = valid && m < g.M ? g.sorted_token_ids[m] : -1;
    }
  };
  auto request_tile = [&](int lid) {   // ahead of set_fetch_tile
    if constexpr (GROUPED) {
      const bool valid = SPLIT ? lid != kNoTile : lid < walk.end;
      m_nxt = n_nxt = 0;
      if (valid) runs.origin(lid, m_nxt, n_nxt);
      load_row_ids(valid, m_nxt);
      int tile_m = g.tile_m;
      asm volatile("" : "+s"(tile_m));
      expert_nxt = g.sorted_expert_ids[m_nxt / tile_m];
    }
  };
  int kq_nxt = KQ;   // K-quads of the tile being fetched
  auto set_fetch_tile = [&](int lid) {
    fetch_valid = SPLIT ? lid != kNoTile : lid < walk.end;
    // a tile that is split along K starts at K-quad q0: folded into the offsets, so that stages count from 0 in every tile
    const bool part = SPLIT && fetch_valid && lid >= walk.end;
    const int qb = part ? walk.quads & 0xFFFF : 0;
    kq_nxt = part ? walk.quads >> 16 : KQ;
    const uint32_t ka0 = (uint32_t)(qb * SPQ * C::A_RB), kb0 = (uint32_t)(qb * SPQ * C::B_RB);
    int m0 = m_nxt, n0 = n_nxt;
    if (!GROUPED && fetch_valid) walk.origin<C::BM>(lid, m0, n0);
    int ln = lane;
    if constexpr (GROUPED) asm volatile("" : "+v"(ln));   // (as in load_row_ids)
    const int row = wn * P::A_RPI + ln / C::A_CPR;   // of the team's 128
    const int a_col0 = ((ln % C::A_CPR) ^ swz<C::A_CPR>(wm0 + row)) * 16, b_row0 = wn0 + ln / C::B_CPR;
    uint32_t row_off[2];   // grouped: where the rows of eid begin in A
    if constexpr (GROUPED) {
      bool any = false;
      int replicas = g.replicas;
      asm volatile("" : "+s"(replicas));
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int id = eid[u];
        const bool ok = id >= 0 && id < g.num_valid_ids;
        any = any || ok;
        row_off[u] = ok ? (uint32_t)((int64_t)(id / replicas) * g.lda) : kOobOffset;
      }
      skip_nxt = __builtin_amdgcn_ballot_w64(any) == 0;
    }
    int expert = 0;
    if constexpr (GROUPED) {
      // an id outside [0, experts) would move the descriptor's base past W, where the range check no longer helps
      expert = __builtin_amdgcn_readfirstlane(expert_nxt);
      expert = expert < 0 ? 0 : (expert >= g.num_experts ? g.num_experts - 1 : expert);
    }
    const uint8_t* Bbase = g.B + (GROUPED ? (int64_t)expert * g.b_expert_stride : 0);
    rsB = make_rsrc(Bbase, operand_bytes(g.N, g.ldb, Kb_b));
#pragma unroll
    for (int q = 0; q < AL; ++q) {
      if constexpr (GROUPED) {
        // (the team's row of instruction q: all of them lie in one half of the 128 when q is known)
        const uint32_t off = __builtin_amdgcn_ds_bpermute(((row + q * 4 * P::A_RPI) & 63) * 4, row_off[q * 4 * P::A_RPI / 64]);
        a_voff[q] = off == kOobOffset ? off : off + a_col0 + ka0;
      } else {
        const int64_t grow = m0 + wm0 + row + q * 4 * P::A_RPI;
        a_voff[q] = fetch_valid && grow < g.M ? (uint32_t)(grow * g.lda + a_col0) + ka0 : kOobOffset;
      }
    }
    if constexpr (TEAM == 1) {
#pragma unroll
      for (int q = 0; q < BL; ++q) {
        const int col = b_col(q, ln);
        const int64_t grow = n0 + b_row0 + q * P::B_RPI;
        b_voff[q] = (fetch_valid && grow < g.N) ? (uint32_t)(grow * g.ldb + col) + kb0 : kOobOffset;
      }
    }
    // a tile that overhangs the matrix reuses the last scale group (its rows are discarded anyway)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int grp = (m0 + wm0) / 64 + u;
      as_nxt[u] = ((grp < a_groups ? grp : a_groups - 1) * KQ + qb) * 1024;
    }
    const int grp = (n0 + wn0) / 64;
    bs_nxt = (GROUPED ? (int)(expert * (g.bs_expert_stride * 4)) : 0) +
             ((grp < b_groups ? grp : b_groups - 1) * KQ + qb) * 1024;
  };
  int kq = KQ;       // K-quads of the tile being computed
  auto nst = [&]() { return SPLIT ? kq * SPQ : nstages; };   // its stages
  // local stage sl of the fetch tile into A buffer abuf / B buffer bbuf; a stage at or beyond nst and the 16-byte chunks
  // beyond the end of K read nothing and zero-fill their LDS bytes (out-of-range buffer offset).  (Walks of several tiles
  // have two stages or more in every tile, so the first two of the next one pass as well; a tile that is split along K has
  // whole stages only: its limits below are those of its first quad, never too small.)
  auto issue_a = [&](int sl, int abuf) {
    lds_u8* const base = smem + abuf * C::A_STAGE + wm0 * C::A_RB + wn * 1024;
    const int ka = sl * C::A_RB;
    const int klim = sl < nst() ? Kb_a - ka : 0;   // bytes of this stage's rows that exist
#pragma unroll
    for (int q = 0; q < AL; ++q) {
      // (without a K tail a stage at or beyond nst is only ever requested once the walk has no further tile, and
      // then every offset is out of range already)
      const uint32_t v = (KTAIL && a_col0 >= klim) ? kOobOffset : a_voff[q];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsA, (lds_void*)(base + q * 4096), 16, v, ka, 0, 0);
    }
  };
  auto issue_b = [&](int sl, int bbuf, int q0 = 0, int q1 = P::BL) {   // DMA instructions q0 .. q1 - 1
    if constexpr (TEAM == 1) {
      lds_u8* const base = smem + P::B_BASE + bbuf * C::B_STAGE + wn0 * C::B_RB;
      const int kb = sl * C::B_RB;
      const int klim = sl < nst() ? Kb_b - kb : 0;
#pragma unroll
      for (int q = q0; q < q1; ++q) {
        const int col = b_col(q, lane);
        const uint32_t v = (KTAIL && col >= klim) ? kOobOffset : b_voff[q];
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsB, (lds_void*)(base + q * 1024), 16, v, kb, 0, 0);
      }
    }
  };

  v4f acc[MT][4];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
  const int swa = swz<C::A_CPR>(r), swb = swz<C::B_CPR>(r);

  // ---- output of a finished tile: lane (c, g) of tile (i, j) holds row 16 i + c, columns
  // 32 (j / 2) + 8 g + 4 (j % 2) .. + 3 (see bperm_tile_off); the accumulators are cleared for the next tile ------------------------------------
  OutT* const Cp = (OutT*)g.C;
  const bool vec_ok = (g.ldc % 4 == 0) && (((uintptr_t)g.C) % 16 == 0);
  // the lane's 8 consecutive outputs of a tile pair as 16-byte stores: every row start 16-byte aligned
  const bool vec8_ok = ((g.ldc * (int64_t)sizeof(OutT)) % 16 == 0) && (((uintptr_t)g.C) % 16 == 0);
  const bool accumulate = g.accumulate != 0;
  auto write_tile = [&](int m0, int n0) {
    if constexpr (!GROUPED) {
      // interior tile, plain store: one address per lane, everything else immediate offsets
      if (m0 + C::BM <= g.M && n0 + 256 <= g.N && vec8_ok && !accumulate) {
        OutT* p = Cp + (int64_t)(m0 + wm0 + r) * g.ldc + (n0 + wn0 + 8 * gq);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
#pragma unroll
          for (int jp = 0; jp < 2; ++jp) {
            store8_full<OutT>(p + 32 * jp, acc[i][2 * jp], acc[i][2 * jp + 1]);
            acc[i][2 * jp] = (v4f){0.f, 0.f, 0.f, 0.f};
            acc[i][2 * jp + 1] = (v4f){0.f, 0.f, 0.f, 0.f};
          }
          p += 16 * g.ldc;
        }
        return;
      }
      // ragged edge, accumulation into C, or C rows that are not 16-byte aligned: the same stores with the rows and
      // columns beyond C masked, still inside the phase.  (A checked writer outside of the kernel body took these
      // tiles before; it was handed the accumulators in scratch memory and waited for each quad in turn, about 50 us
      // for a tile: 1531 x 14336 x 4096 MXFP8 took 145 us against 92 us for 1536 rows.)
      OutT* p = Cp + (int64_t)(m0 + wm0 + r) * g.ldc + (n0 + wn0 + 8 * gq);
      const int rows = g.M - (m0 + wm0 + r), cols = g.N - (n0 + wn0 + 8 * gq);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        if (16 * i < rows) {
#pragma unroll
          for (int jp = 0; jp < 2; ++jp) {
            if (accumulate) add8_edge<OutT>(p + 32 * jp, acc[i][2 * jp], acc[i][2 * jp + 1], cols - 32 * jp);
            store8_edge<OutT>(p + 32 * jp, acc[i][2 * jp], acc[i][2 * jp + 1], cols - 32 * jp);
          }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
        p += 16 * g.ldc;
      }
      return;
    }
    // grouped: row 16 i + c of the team's half goes to row `id` of C, where id is the routed-slot index
    // that lane 16 (i % 4) + c of eid[i / 4] has held since the tile began (no load latency here)
    const bool cols_in = n0 + 256 <= g.N && vec8_ok && !accumulate;   // uniform
    float ewt[2] = {1.f, 1.f};
    if (g.topk_weights) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (eid[u] >= 0 && eid[u] < g.num_valid_ids) ewt[u] = g.topk_weights[eid[u]];
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int src = (16 * (i & 3) + r) * 4;
      const int id = __builtin_amdgcn_ds_bpermute(src, eid[i >> 2]);
      const bool ok = id >= 0 && id < g.num_valid_ids;
      float w = 1.f;
      if (g.topk_weights) w = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(src, __builtin_bit_cast(int, ewt[i >> 2])));
      OutT* const p = Cp + (int64_t)id * g.ldc + (n0 + wn0 + 8 * gq);
      if (cols_in) {
        if (ok) {
#pragma unroll
          for (int jp = 0; jp < 2; ++jp) store8_full<OutT>(p + 32 * jp, acc[i][2 * jp] * w, acc[i][2 * jp + 1] * w);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int n = n0 + wn0 + 8 * gq + bperm_tile_off(j);
          if (ok && n < g.N)
            store4<OutT>(p + bperm_tile_off(j), acc[i][j] * w, accumulate, g.N - n, vec_ok);
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
    }
  };
  // ---- prologue: stages 0 and 1 of the first tile, scales of its K-quad 0 ---------------------------------
  // (without SPLIT the walk is the arithmetic sequence alone)
  auto next = [&](int t) { return SPLIT ? walk.next(t) : t + walk.step; };
  int lid = SPLIT ? walk.head() : walk.first;   // tile being computed
  // the one before tile t: the tail follows the workgroup's tile of the last whole round
  auto before = [&](int t) { return (SPLIT && t >= walk.end ? walk.end + ((int)blockIdx.x >> 3) : t) - walk.step; };
  request_tile(lid);
  set_fetch_tile(lid);
  kq = kq_nxt;
  issue_a(0, 0);
  issue_b(0, 0);
  issue_a(1, 1);
  issue_b(1, 1);
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  if constexpr (TEAM == 1) asm volatile("s_barrier" ::: "memory");   // one phase behind team 0
  __builtin_amdgcn_sched_barrier(0);

  int abuf = 0, abuf2 = 2, bbuf = 0;   // buffers of stage s (A, B) and of stage s + 2 (A)
  int Q = 0;
  auto stage = [&](auto t0c) {
    constexpr int t0 = decltype(t0c)::value;
    const int s = Q * SPQ + t0 / C::KSUB;
    if (s >= nst()) return;
    // =============================== memory phase ==================================================
    if constexpr (t0 == 0) {
      // Scales of this K-quad, first in the queue of this memory phase: they have the whole phase to arrive, and
      // the MFMA phase holds no vector-memory instruction at all.  (Requested a stage ahead, stage by stage, in
      // 4-byte loads, they arrive no earlier in effect: what they cost is their share of the address unit, which
      // three 16-byte loads per quad keep smallest.)
      load_scales(as_cur, bs_cur, Q);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (t0 == 0) {
      if (s == 0 && lid != walk.first && (!SPLIT || walk.first < walk.end)) {
        // the previous tile's output leaves while the other team is in its MFMA phase
        // (the tile index passes through an opaque move: otherwise the compiler computes the eight row
        // pointers of the stores when the tile begins and keeps them in registers through all its stages)
        int plid = before(lid);   // (always a whole tile: a split one is the last of the walk)
        asm volatile("" : "+s"(plid));
        int pm0 = 0, pn0 = n_out;   // (grouped rows are placed by their ids)
        if constexpr (!GROUPED) walk.origin<C::BM>(plid, pm0, pn0);
        write_tile(pm0, pn0);
      }
    }
    if (GROUPED && t0 == 0 && Q == (nst() > 3 ? (nst() - 3) / SPQ : 0)) request_tile(next(lid));
    // from stage nst - 2 on, the loads run ahead into the next tile of the walk
    if (s + 2 == nst()) set_fetch_tile(next(lid));
    if (GROUPED && s + 1 == nst()) load_row_ids(true, m_cur);
    const bool wrapped = s + 2 >= nst();
    const int sl = wrapped ? s + 2 - nst() : s + 2;   // local stage the loads fetch
    const int sl_eff = (wrapped && (!fetch_valid || nst() < 2)) ? nst() : sl;
    lds_u8* const atile = smem + abuf * C::A_STAGE + (wm0 + r) * C::A_RB;
    lds_u8* const btile = smem + P::B_BASE + bbuf * C::B_STAGE + (wn0 + bperm_lane_off(r)) * C::B_RB;
    issue_a(sl_eff, abuf2);
    v8i bf[C::KSUB][4], af[C::KSUB][MT];
    if (!(GROUPED && skip_cur)) {
      // B tiles 0, 1 (rows 0 .. 31 of the wave's 64), then tiles 2, 3, then the early A tiles: LDS returns reads in
      // order, so the DMA that refills the first half of the B rows can go as soon as the first group is back
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int kk = 0; kk < C::KSUB; ++kk)
#pragma unroll
          for (int j = 2 * h; j < 2 * h + 2; ++j) bf[kk][j] = load_frag<C::B_RB, C::B_EB>(btile, bperm_tile_off(j), kk, gq, swb);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int kk = 0; kk < C::KSUB; ++kk)
#pragma unroll
        for (int i = 0; i < EARLY; ++i) af[kk][i] = load_frag<C::A_RB, C::A_EB>(atile, 16 * i, kk, gq, swa);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (TEAM == 1) {
      // the B buffer of this stage is free once this wave's own reads have returned
      constexpr int NBH = 2 * C::KSUB * (C::B_EB == 8 ? 2 : 1);       // LDS reads of two B tiles
      constexpr int NAE = EARLY * C::KSUB * (C::A_EB == 8 ? 2 : 1);   // LDS reads of the early A tiles
      asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(NBH + NAE) : "memory");
      __builtin_amdgcn_sched_barrier(0);
      issue_b(sl_eff, bbuf, 0, BL / 2);
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(NAE) : "memory");
      __builtin_amdgcn_sched_barrier(0);
      issue_b(sl_eff, bbuf, BL / 2, BL);
      // everything older than this phase's loads has landed: A and B of stage s + 1 (the scale loads issued
      // at the start of this phase are younger than those and may stay in flight; the MFMA phase waits for them)
      constexpr int younger = (t0 == 0) ? NSC : 0;
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(AL + BL + younger));
    }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // fragments are in registers
    __builtin_amdgcn_sched_barrier(0);
    // =============================== MFMA phase ====================================================
    __builtin_amdgcn_s_setprio(1);
    auto read_pair = [&](int i0) {
#pragma unroll
      for (int kk = 0; kk < C::KSUB; ++kk)
#pragma unroll
        for (int i = i0; i < i0 + 2; ++i) {
          af[kk][i] = load_frag<C::A_RB, C::A_EB>(atile, 16 * i, kk, gq, swa);
        }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto mfma_pair = [&](int i0, int n = 2) {   // row tiles i0 .. i0 + n - 1
#pragma unroll
      for (int kk = 0; kk < C::KSUB; ++kk) {
#pragma unroll
        for (int i = i0; i < i0 + n; ++i) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            acc[i][j] = mfma_scaled<C::BF, C::AF>(bf[kk][j], af[kk][i], acc[i][j], j, sb[t0 + kk], (at0 + i) % 4,
                                                  sa[(at0 + i) / 4][t0 + kk]);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    // A tiles below EARLY were read in the memory phase; the rest is read EARLY * 4 MFMAs ahead of use
    if (!(GROUPED && skip_cur)) {
#pragma unroll
      for (int ip = 0; ip < MT; ip += 2) {
        if (ip == 0) {
          // the phase opens with MFMAs, not with LDS read issue: the matrix pipe restarts that much sooner after the
          // hand-over, and the reads issue while the first MFMAs run
          mfma_pair(0, 1);
          read_pair(EARLY);
          mfma_pair(1, 1);
          continue;
        }
        if (ip + EARLY < MT) read_pair(ip + EARLY);
        mfma_pair(ip);
      }
    }
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (TEAM == 0) {
      // A of stage s + 1 (issued one stage ago) must have landed; A of stage s + 2 may stay in flight
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(AL));
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    abuf = abuf == 2 ? 0 : abuf + 1;
    abuf2 = abuf2 == 2 ? 0 : abuf2 + 1;
    bbuf ^= 1;
  };
  for (; SPLIT ? lid != kNoTile : lid < walk.end; lid = next(lid)) {
    skip_cur = skip_nxt;
    n_out = n_cur;
    m_cur = m_nxt; n_cur = n_nxt;
    kq = kq_nxt;
    as_cur[0] = as_nxt[0];
    as_cur[1] = as_nxt[1];
    bs_cur = bs_nxt;
    for (Q = 0; Q < kq; ++Q) {
      stage(std::integral_constant<int, 0>{});
      if constexpr (C::KSUB == 1) stage(std::integral_constant<int, 1>{});
      stage(std::integral_constant<int, 2>{});
      if constexpr (C::KSUB == 1) stage(std::integral_constant<int, 3>{});
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // trailing zero-fill DMA has left the queue
  __builtin_amdgcn_sched_barrier(0);
  if (!SPLIT || walk.tail == kNoTile) {
    int pm0 = m_cur, pn0 = n_cur;
    if constexpr (!GROUPED) walk.origin<C::BM>(SPLIT ? walk.first + (walk.end - 1 - walk.first) / walk.step * walk.step : lid - walk.step, pm0, pn0);
    write_tile(pm0, pn0);
  } else {
    // partial sums, as the lanes hold them: 1 KiB per store instruction
    v4f* const t = (v4f*)g.tail + ((int64_t)blockIdx.x * 8 + TEAM * 4 + wn) * 32 * 64 + lane;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) t[(i * 4 + j) * 64] = acc[i][j];
  }
  if constexpr (TEAM == 0) asm volatile("s_barrier" ::: "memory");   // pairs with team 1's extra barrier
}

// rows of C (slots, when grouped) that have tiles
template <bool GROUPED>
__device__ __forceinline__ int pp_rows(const GemmArgs& g) {
  if constexpr (GROUPED) {
    if (g.num_slots) {
      const int n = *g.num_slots;
      return n < 0 ? 0 : n < g.M ? n : g.M;
    }
  }
  return g.M;
}
template <class C, bool GROUPED, bool SPLIT>
__device__ __forceinline__ TileWalk pp_walk(const GemmArgs& g) {
  const int M = pp_rows<GROUPED>(g);
  if constexpr (SPLIT) return make_split_walk(M, g.N, g.K / 512, C::KSUB == 2);
  else return make_tile_walk(M, g.N, C::BM);
}

template <class C, typename OutT, bool GROUPED, bool SPLIT>
__global__ __launch_bounds__(512) void gemm_pp_kernel(const GemmArgs g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem_generic[];
  lds_u8* const smem = (lds_u8*)smem_generic;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  const int ksteps = (g.K + 127) / 128;
  const TileWalk walk = pp_walk<C, GROUPED, SPLIT>(g);
  if (walk.head() == kNoTile) return;   // uniform: nothing left for this workgroup
  // (uniform.  The MXFP4 instance keeps the one masked body: a second, unmasked one measured no faster on it.)
  // (a split K is a whole number of K-quads)
  const bool ktail = C::KSUB != 1 || (!SPLIT && (g.K % 128 != 0 || ksteps < 2));
  if (ktail) {
    if (wave < 4)
      pp_body<C, OutT, GROUPED, SPLIT, 0, true>(g, smem, wave, lane, walk);
    else
      pp_body<C, OutT, GROUPED, SPLIT, 1, true>(g, smem, wave - 4, lane, walk);
  } else if constexpr (C::KSUB == 1) {
    if (wave < 4)
      pp_body<C, OutT, GROUPED, SPLIT, 0, false>(g, smem, wave, lane, walk);
    else
      pp_body<C, OutT, GROUPED, SPLIT, 1, false>(g, smem, wave - 4, lane, walk);
  }
}

// Adds up the partial sums of the tiles that gemm_pp_kernel split along K, in the order of their slices, and writes them.
// Workgroup: (XCD, one of its split tiles, one wave's 128 x 64 block of it), four waves of two row tiles each.
template <class C, typename OutT, bool GROUPED>
__global__ __launch_bounds__(256) void pp_tail_kernel(const GemmArgs g, const int grid) {
  const int xcd = blockIdx.x & 7, wv = (blockIdx.x >> 3) & 7, at = blockIdx.x >> 6;
  const int lane = threadIdx.x & 63, r = lane & 15, gq = lane >> 4, w4 = threadIdx.x >> 6;
  TileWalk walk = {};
  walk.tiles_m = (pp_rows<GROUPED>(g) + 255) / 256;
  walk.tiles_n = (g.N + 255) / 256;
  const XcdShare x = xcd_share(walk.tiles_m * walk.tiles_n, grid, xcd);
  const int rest = x.count % x.wgs, S = tail_splits(rest, x.wgs, g.K / 512, C::KSUB == 2);
  if (S == 1 || at >= rest) return;
  int m0, n0;
  if constexpr (GROUPED) {
    ExpertRuns runs = {g.sorted_expert_ids, g.tile_m, walk.tiles_m, walk.tiles_n};
    runs.origin(x.start + x.count - rest + at, m0, n0);
  } else {
    walk.origin(x.start + x.count - rest + at, m0, n0);
  }
  const int n = n0 + (wv & 3) * 64 + 8 * gq;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int i = w4 * 2 + u, m = m0 + (wv >> 2) * 128 + 16 * i + r;
    v4f v[4] = {};
    for (int s = 0; s < S; ++s) {
      const int wg = (at * S + s) * 8 + xcd;
      const v4f* const t = (const v4f*)g.tail + ((int64_t)wg * 8 + wv) * 32 * 64 + i * 4 * 64 + lane;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] += t[j * 64];
    }
    int64_t row = m;
    bool ok = m < g.M;
    float w = 1.f;
    if constexpr (GROUPED) {
      const int id = ok ? g.sorted_token_ids[m] : -1;
      ok = id >= 0 && id < g.num_valid_ids;
      row = id;
      if (ok && g.topk_weights) w = g.topk_weights[id];
    }
    if (!ok) continue;
    OutT* const p = (OutT*)g.C + row * g.ldc + n;
#pragma unroll
    for (int jp = 0; jp < 2; ++jp) {
      v4f v0 = v[2 * jp], v1 = v[2 * jp + 1];
      if constexpr (GROUPED) { v0 *= w; v1 *= w; }
      if (g.accumulate) add8_edge<OutT>(p + 32 * jp, v0, v1, g.N - n - 32 * jp);
      store8_edge<OutT>(p + 32 * jp, v0, v1, g.N - n - 32 * jp);
    }
  }
}

template <class C, typename OutT, bool GROUPED, bool SPLIT>
int launch_pp(const GemmArgs& g, hipStream_t stream) {
  auto kern = gemm_pp_kernel<C, OutT, GROUPED, SPLIT>;
  static int attr_done = 0;   // benign race: the attribute call is idempotent
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       PP<C>::LDS_BYTES);
    if (e != hipSuccess)
      return set_error(MX_ERR_LAUNCH, "hipFuncSetAttribute(%d bytes LDS): %s", PP<C>::LDS_BYTES,
                       hipGetErrorString(e));
    attr_done = 1;
  }
  int64_t grid = pp_grid(g.M, g.N, g.K, C::KSUB, C::BM);
  if (grid <= 0) return MX_OK;
  if (SPLIT) grid = num_cus();   // idle workgroups of a single, partly filled round take part too
  hipError_t e = launch_kernel(kern, dim3((unsigned)grid), dim3(512), PP<C>::LDS_BYTES, stream, g);
  if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "gemm_pp_kernel launch: %s", hipGetErrorString(e));
  if constexpr (SPLIT) {
    e = launch_kernel(pp_tail_kernel<C, OutT, GROUPED>, dim3(8 * 8 * kTailMax), dim3(256), 0, stream, g, (int)grid);
    if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "pp_tail_kernel launch: %s", hipGetErrorString(e));
  }
  return MX_OK;
}

}  // namespace

// One element-format pair (grouped and plain, fp32 and bf16 output) per compilation of this file, so that the pairs
// build in parallel: MX_PP_PAIR names it.
template <int AF, int BF>
int launch_pp_pair(const GemmArgs& g, hipStream_t stream) {
  using C = Cfg<AF, BF, 256, 256, 2, 4>;
  const bool grouped = g.sorted_token_ids != nullptr;
  auto run = [&](auto split) {
    constexpr bool S = decltype(split)::value;
    if (g.c_dtype == MX_F32)
      return grouped ? launch_pp<C, float, true, S>(g, stream) : launch_pp<C, float, false, S>(g, stream);
    return grouped ? launch_pp<C, uint16_t, true, S>(g, stream) : launch_pp<C, uint16_t, false, S>(g, stream);
  };
  if (g.tile_rows == 192 && !grouped) {
    using C192 = Cfg<AF, BF, 192, 256, 2, 4>;
    return g.c_dtype == MX_F32 ? launch_pp<C192, float, false, false>(g, stream) : launch_pp<C192, uint16_t, false, false>(g, stream);
  }
  return g.tail ? run(std::true_type{}) : run(std::false_type{});
}
#if MX_PP_PAIR == 0
template int launch_pp_pair<MX_E4M3, MX_E4M3>(const GemmArgs&, hipStream_t);
extern template int launch_pp_pair<MX_E5M2, MX_E5M2>(const GemmArgs&, hipStream_t);
extern template int launch_pp_pair<MX_E2M1, MX_E2M1>(const GemmArgs&, hipStream_t);
extern template int launch_pp_pair<MX_E4M3, MX_E2M1>(const GemmArgs&, hipStream_t);

int launch_gemm_pingpong(const GemmArgs& g, hipStream_t stream) {
  if (g.c_dtype != MX_F32 && g.c_dtype != MX_BF16)
    return set_error(MX_ERR_DTYPE, "MFMA kernel: output dtype %d not supported", g.c_dtype);
#define MX_CASE(AFMT, BFMT) \
  if (g.a_fmt == AFMT && g.b_fmt == BFMT) return launch_pp_pair<AFMT, BFMT>(g, stream);
  MX_CASE(MX_E4M3, MX_E4M3)
  MX_CASE(MX_E5M2, MX_E5M2)
  MX_CASE(MX_E2M1, MX_E2M1)
  MX_CASE(MX_E4M3, MX_E2M1)
#undef MX_CASE
  return set_error(MX_ERR_DTYPE, "MFMA kernel: unsupported element format pair (%d, %d)", g.a_fmt,
                   g.b_fmt);
}
#elif MX_PP_PAIR == 1
template int launch_pp_pair<MX_E5M2, MX_E5M2>(const GemmArgs&, hipStream_t);
#elif MX_PP_PAIR == 2
template int launch_pp_pair<MX_E2M1, MX_E2M1>(const GemmArgs&, hipStream_t);
#else
template int launch_pp_pair<MX_E4M3, MX_E2M1>(const GemmArgs&, hipStream_t);
#endif

}  // namespace mx
