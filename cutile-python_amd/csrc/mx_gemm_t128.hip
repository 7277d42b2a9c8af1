// 128 x 128 one-tile block-scaled GEMM (gfx950), four waves of 64 x 64.  Same math, operand layouts, LDS swizzle and column
// order as mx_gemm_mfma.hip; what differs is the schedule.
//
// What bounded the lock-step kernel that ran these products before was latency: with one workgroup on a CU a stage
// took 2150 cycles for 512 cycles of MFMA (1024 x 4096 x 4096 MXFP8, SQ_BUSY_CYCLES 69 k for 32 stages; with two
// workgroups on the CU 77 k for twice the work), one chain of load wait, barrier, fragment reads and MFMAs after another.
// Here the fragments of stage s + 1 are read into a second register set while the MFMAs of stage s run, behind one
// barrier per stage, and the LDS-DMA runs NS stages ahead:
//   iteration s:  wait until stage s + 1 has landed; barrier (everybody's part has landed, everybody has read stage s)
//                 issue the DMA of stage s + NS into the buffer of stage s (more than two stages: between the MFMAs, SPREAD)
//                 16 (32) MFMAs of stage s, the fragment reads of stage s + 1 between them
// (order of the requests and what the waits count: mx_t128_schedule.h).
// 64 x 64 tiles (four waves of 32 x 32, eight stages in flight or four) take products that leave CUs idle: a stage is 0.25 us
// instead of 0.62, and there are four times as many workgroups.  Six products 200 x 328 x 992 with an addend 10.7 -> 7.0 us,
// 1024 x 1024 x 4096 21.4 -> 13.4 (19.2 with K split four ways), 256 x 4096 x 8192 22.7 (split) -> 20.5; with two workgroups
// on a CU 512 x 4096 x 4096 22.4 -> 17.1; beyond that the larger tile reads less (1200 x 2048 x 2048 14.6 against 15.7).
//
// NS = 4 (128 KiB, one workgroup per CU) for grids that leave CUs with one tile, NS = 2 (64 KiB) where two workgroups share
// a CU.  The fragment reads (64 KiB per stage at 128 bytes per clock) are as long as the MFMAs of a stage, so a CU can get
// to about half of the MFMA rate; larger products go to the 256 x 256 kernel.
//
// Scales: the native layout, or (a_plain / b_plain) the caller's K-contiguous rows as they are, 16 bytes of a row per
// K-quad, of which a lane keeps its own byte of each K-step, four in one register, which the instruction's byte select
// walks.  That saves small products the re-layout launch in front of them.  Rows at any byte (kScaleAny: K / 32 no multiple of
// four in a dense tensor, or a K that ends inside a stage) cannot come by DMA: a wave's lanes fetch the five aligned dwords
// around their 16 bytes, shift them into place, clear what lies beyond K and write them to the same LDS slots, a quad
// ahead.  Six products 200 x 328 x 992 15.6 -> 11.9 us (re-layout
// 4.5 us and the wait for it), a list of 24 of 96 .. 1536 42.2 -> 35.6.
#include <type_traits>

#include "mx_gemm_pp.h"
#include "mx_gemm_t128.h"
#include "mx_gemm_tile.h"
#include "mx_t128_schedule.h"

namespace mx {
namespace {

// where an operand's scales are: native layout; plain rows that the DMA can fetch; plain rows at any byte (both operands)
constexpr int kScaleNative = 0, kScalePlain = 1, kScaleAny = 2;

// A stage's requests go out between its MFMAs: all four waves' at once behind the barrier they keep the address unit busy for some
// 500 cycles, the length of a stage's MFMAs, in which none of these is issued.  2048 x 2048 x 2048 FP8 15.2 -> 13.5 us, x 8192 43.0 ->
// 40.9, FP4 26.9 -> 25.3, 200 x 14336 x 4096 24.3 -> 23.0; on tiles of 64 0 - 6 % (packed scales, 300 x 2000 x 7168 FP8
// 18.4 -> 17.8, FP4 weights 16.8 -> 15.8, with two workgroups on a CU 1400 x 1400 x 8192 29.8 -> 28.8; plain ones 900 x 900 x 8192 21.1 ->
// 20.9).  Not with two stages, where a later request is a later stage (512 x 14336 x 4096 35.8 -> 39.6), nor beside the larger tile's
// scales through registers (1111 x 2100 x 4032 21.6 -> 22.2), nor beside those of the smaller one where eight stages are in flight for long
// (t128_any_spread).
template <class C, int NS, int AS>
constexpr bool kSpread = NS > 2 && !(AS == kScaleAny && C::BM == 128);

template <class C, int NS, int AS, int BS, bool GROUPED, bool SPREAD = kSpread<C, NS, AS>>
__device__ __forceinline__ void t128_tile(const T128Args& g, lds_u8* const smem, const int pid, const int split, const int bz) {
  constexpr int KS = C::KSUB, SPQ = 4 / KS, MT = C::MT, NT = C::NTL;
  constexpr bool AP = AS != kScaleNative, BP = BS != kScaleNative, ANY = AS == kScaleAny;
  static_assert(ANY == (BS == kScaleAny) && !(ANY && GROUPED) && MT == NT && (C::BM == 128 || !GROUPED), "");
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, gq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave >> 1) * C::WTM, wn0 = (wave & 1) * C::WTN;

  // ---- tile of C: XCD-aware, then grouped along M (as in mx_gemm_mfma.hip) ------------------------------------------
  const int tiles_m = (g.M + C::BM - 1) / C::BM, tiles_n = (g.N + C::BN - 1) / C::BN;
  int m0, n0;
  {
    const int total = tiles_m * tiles_n;
    const int xcd = pid & 7, loc = pid >> 3, per = total >> 3, rem = total & 7;
    const int lid = xcd * per + (xcd < rem ? xcd : rem) + loc;
    constexpr int GM = 4;
    const int in_group = GM * tiles_n;
    const int gid = lid / in_group, first_m = gid * GM;
    const int gsz = (tiles_m - first_m) < GM ? (tiles_m - first_m) : GM;
    const int in = lid % in_group;
    m0 = (first_m + in % gsz) * C::BM;
    n0 = (in / gsz) * C::BN;
  }
  int expert = 0;
  if constexpr (GROUPED) {
    expert = g.sorted_expert_ids[m0 / g.tile_m];
    expert = expert < 0 ? 0 : (expert >= g.num_experts ? g.num_experts - 1 : expert);
  }
  // K-quads of this split
  const int ksteps = (g.K + 127) / 128, KQ = (ksteps + 3) / 4;
  const int q0 = (int)((int64_t)split * KQ / g.k_splits), q1 = (int)((int64_t)(split + 1) * KQ / g.k_splits);
  const int nst = (ksteps + KS - 1) / KS, s0 = q0 * SPQ, s1 = q1 * SPQ < nst ? q1 * SPQ : nst;   // stages [s0, s1)

  const uint8_t* const Ab = g.A + (int64_t)bz * g.a_batch;
  const uint8_t* const Bb = g.B + (int64_t)bz * g.b_batch + (GROUPED ? (int64_t)expert * g.b_expert : 0);
  const int64_t a_rows = GROUPED ? g.a_rows : g.M;
  const __amdgpu_buffer_rsrc_t rsA = make_rsrc(Ab, operand_bytes(a_rows, g.lda, (int64_t)g.K * C::A_EB / 8));
  const __amdgpu_buffer_rsrc_t rsB = make_rsrc(Bb, operand_bytes(g.N, g.ldb, (int64_t)g.K * C::B_EB / 8));
  const __amdgpu_buffer_rsrc_t rsAs =
      make_rsrc(g.As + (int64_t)bz * g.as_batch,
                AP ? operand_bytes(a_rows, g.ldas, g.K / 32) : (uint32_t)(packed_scale_dwords(g.M, g.K) * 4));
  const __amdgpu_buffer_rsrc_t rsBs =
      make_rsrc(g.Bs + (int64_t)bz * g.bs_batch + (GROUPED ? (int64_t)expert * g.bs_expert : 0),
                BP ? operand_bytes(g.N, g.ldbs, g.K / 32) : (uint32_t)(packed_scale_dwords(g.N, g.K) * 4));

  // ---- DMA: instruction q of wave w fills 1 KiB of the stage: rows (q * 4 + w) * RPI ... ------------------------------
  constexpr int AL = C::A_LOADS, BL = C::B_LOADS, TL = AL + BL;
  constexpr int ARPI = 64 / C::A_CPR, BRPI = 64 / C::B_CPR;
  uint32_t avo[AL], bvo[BL];
  const int a_lr = lane / C::A_CPR, b_lr = lane / C::B_CPR;
  // (rows of different instructions of a wave differ by a multiple of 32: the same swizzle, hence the same column)
  const int a_col = ((lane % C::A_CPR) ^ swz<C::A_CPR>(wave * ARPI + a_lr)) * 16;
  const int b_col = ((lane % C::B_CPR) ^ swz_bperm<C::B_CPR>(wave * BRPI + b_lr)) * 16;
#pragma unroll
  for (int q = 0; q < AL; ++q) {
    int64_t row = m0 + (q * 4 + wave) * ARPI + a_lr;
    bool ok = row < g.M;
    if constexpr (GROUPED) {
      const int id = ok ? g.sorted_token_ids[row] : 0x7FFFFFFF;
      ok = ok && id >= 0 && id < g.num_valid_ids;
      row = id / g.replicas;
    }
    avo[q] = ok ? (uint32_t)(row * g.lda + a_col) : kOobOffset;
  }
#pragma unroll
  for (int q = 0; q < BL; ++q) {
    const int64_t row = n0 + (q * 4 + wave) * BRPI + b_lr;
    bvo[q] = row < g.N ? (uint32_t)(row * g.ldb + b_col) : kOobOffset;
  }
  const int Ka = g.K * C::A_EB / 8, Kb = g.K * C::B_EB / 8;   // bytes of a row
  // part `part` of `parts` of stage s; a stage at or beyond s1 and the chunks beyond the end of K arrive as zeros
  auto issue = [&](int s, int buf, int part, int parts) {
    lds_u8* const base = smem + buf * C::STAGE + wave * 1024;
    const int ka = s * C::A_RB, kb = s * C::B_RB;
    const bool la = s < s1 && a_col < Ka - ka, lb = s < s1 && b_col < Kb - kb;
#pragma unroll
    for (int q = part * AL / parts; q < (part + 1) * AL / parts; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsA, (lds_void*)(base + q * 4096), 16, la ? avo[q] : kOobOffset, ka, 0, 0);
#pragma unroll
    for (int q = part * BL / parts; q < (part + 1) * BL / parts; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsB, (lds_void*)(base + C::A_STAGE + q * 4096), 16, lb ? bvo[q] : kOobOffset, kb,
                                               0, 0);
  };

  // ---- scales: 64 rows (group) x 16 bytes per wave and K-quad, by LDS-DMA SD quads ahead: waves 0, 1 fetch A's two groups,
  // 2, 3 B's.  (Each wave loading what it needs into registers is eight times as many load instructions for plain
  // scales; 1024 x 4096 x 4096 27.2 us that way.)
  using Sched = T128Schedule<NS, SPQ, TL>;
  static_assert(t128_covered<Sched>(), "a wait does not cover what is read behind it");
  constexpr int SD = Sched::SD, SSLOT = 4096;
  lds_u8* const sbase = smem + NS * C::STAGE;
  uint32_t sco;                       // lane offset of this wave's group
  {
    const bool is_b = wave >= 2;
    const int row0 = (is_b ? n0 : m0) + 64 * (wave & 1), rows = is_b ? g.N : g.M;
    const bool plain = is_b ? BP : AP;
    if (C::BM == 64 && (wave & 1)) {   // one group per operand
      sco = kOobOffset;
    } else if (plain) {
      int64_t row = row0 + lane;
      bool ok = row < rows;
      if constexpr (GROUPED) {
        if (!is_b) {
          const int id = ok ? g.sorted_token_ids[row] : 0x7FFFFFFF;
          ok = ok && id >= 0 && id < g.num_valid_ids;
          row = id / g.replicas;
        }
      }
      sco = ok ? (uint32_t)(row * (is_b ? g.ldbs : g.ldas)) : kOobOffset;
    } else {
      sco = row0 / 64 < (rows + 63) / 64 ? (uint32_t)(row0 / 64 * KQ * 1024 + lane * 16) : kOobOffset;
    }
  }
  // kScaleAny: the wave's group through registers
  __amdgpu_buffer_rsrc_t rsAny;
  uint32_t raw[Sched::kAnyLoads], shift = 0;
  if constexpr (ANY) {
    const bool is_b = wave >= 2;
    const uintptr_t at = (uintptr_t)(is_b ? g.Bs + (int64_t)bz * g.bs_batch : g.As + (int64_t)bz * g.as_batch);
    const uint32_t mis = (uint32_t)(at & 3);         // whole dwords: never more than 3 bytes either side of the tensor's own
    rsAny = make_rsrc((const void*)(at - mis), (operand_bytes(is_b ? g.N : g.M, is_b ? g.ldbs : g.ldas, g.K / 32) + mis + 3) & ~3u);
    if (sco != kOobOffset) {
      shift = (sco + mis) & 3;
      sco = (sco + mis) & ~3u;
    }
  }
  auto load_any = [&](int Q) {
    const uint32_t v = Q < q1 ? sco + Q * 16 : kOobOffset;
#pragma unroll
    for (int i = 0; i < Sched::kAnyLoads; ++i) raw[i] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rsAny, v + 4 * i, 0, 0);
  };
  auto store_any = [&](int Q) {
    uint32_t d[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) d[t] = __builtin_amdgcn_alignbyte(raw[t + 1], raw[t], shift);
    if (Q == KQ - 1) {                               // uniform: the next row's bytes are not this one's scales
      const int left = g.K / 32 - 16 * Q;
#pragma unroll
      for (int t = 0; t < 4; ++t) d[t] &= left >= 4 * t + 4 ? ~0u : left <= 4 * t ? 0u : (1u << (8 * (left - 4 * t))) - 1;
    }
    typedef __attribute__((address_space(3))) v4i lds_w4i;
    *(lds_w4i*)(sbase + Q % (SD + 1) * SSLOT + wave * 1024 + lane * 16) = (v4i){(int)d[0], (int)d[1], (int)d[2], (int)d[3]};
  };
  auto load_scales = [&](int Q) {
    lds_u8* const dst = sbase + Q % (SD + 1) * SSLOT + wave * 1024;
    const uint32_t v = Q < q1 ? sco : kOobOffset;
    if (wave < 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsAs, (lds_void*)dst, 16, v, Q * (AP ? 16 : 1024), 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsBs, (lds_void*)dst, 16, v, Q * (BP ? 16 : 1024), 0, 0);
  };
  int sa[4] = {}, sb[4] = {}, san[4] = {}, sbn[4] = {};   // plain: register = tile, byte = K-step; packed: register = K-step, byte = tile
  // plain: the lane's byte gq of each of a row's four dwords
  const uint32_t sel = 0x0c0c0400u + (uint32_t)gq * 0x0101u;
  auto own = [&](const v4i v) {
    const uint32_t lo = __builtin_amdgcn_perm((uint32_t)v.y, (uint32_t)v.x, sel), hi = __builtin_amdgcn_perm((uint32_t)v.w, (uint32_t)v.z, sel);
    return (int)(lo | (hi << 16));
  };
  auto read_scales = [&](int Q) {
    lds_u8* const ta = sbase + Q % (SD + 1) * SSLOT + (AP ? wm0 : wm0 / 64 * 64) * 16;
    lds_u8* const tb = sbase + Q % (SD + 1) * SSLOT + 2048 + (BP ? wn0 : wn0 / 64 * 64) * 16;
    // (packed: a register holds the group's four tiles of a K-step; a wave of 32 rows has the first or the last two)
    if constexpr (AP) {
#pragma unroll
      for (int i = 0; i < MT; ++i) san[i] = own(*(lds_v4i*)(ta + (16 * i + r) * 16));
    } else {
      const v4i v = *(lds_v4i*)(ta + lane * 16);
#pragma unroll
      for (int i = 0; i < 4; ++i) san[i] = MT == 4 ? v[i] : (int)((uint32_t)v[i] >> (wm0 / 2));
    }
    if constexpr (BP) {
#pragma unroll
      for (int j = 0; j < NT; ++j) sbn[j] = own(*(lds_v4i*)(tb + bperm_row(j, r) * 16));
    } else {
      const v4i v = *(lds_v4i*)(tb + lane * 16);
#pragma unroll
      for (int j = 0; j < 4; ++j) sbn[j] = NT == 4 ? v[j] : (int)((uint32_t)v[j] >> (wn0 / 2));
    }
  };
  auto take_scales = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) { sa[i] = san[i]; sb[i] = sbn[i]; }
  };

  v4f acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
  v8i af[2][KS][MT], bf[2][KS][NT];
  const int swa = swz<C::A_CPR>(r), swb = swz<C::B_CPR>(r);
  auto read_a = [&](int buf, auto set, int i) {
    lds_u8* const t = smem + buf * C::STAGE + (wm0 + r) * C::A_RB;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) af[decltype(set)::value][kk][i] = load_frag<C::A_RB, C::A_EB>(t, 16 * i, kk, gq, swa);
  };
  auto read_b = [&](int buf, auto set, int j) {
    lds_u8* const t = smem + buf * C::STAGE + C::A_STAGE + (wn0 + bperm_lane_off(r)) * C::B_RB;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) bf[decltype(set)::value][kk][j] = load_frag<C::B_RB, C::B_EB>(t, bperm_tile_off(j), kk, gq, swb);
  };

  // the fp32 addend (its own operand, or C): every load is requested before the first is waited for, with offsets beyond
  // the matrix for what does not exist.  (One guarded load after another, as for the rows below that are not whole
  // 16-byte pieces, the addend cost more than the product: six 200 x 328 x 992 took 17 us instead of 9.)  Tiles of 64 have
  // the registers to request it ahead of everything else.
  constexpr bool EARLY_ADD = C::BM == 64;
  const int n = n0 + wn0 + 8 * gq;
  const int cols = g.N - n;
  v4f add[GROUPED ? 1 : MT][NT];
  bool added = false;
  auto load_addend = [&]() {
    if constexpr (!GROUPED) {
      const float* const addend = g.acc ? g.acc + (int64_t)bz * g.c_batch
                                  : g.accumulate ? (const float*)g.C + (int64_t)bz * g.c_batch : nullptr;
      const int64_t ld = g.ldc;
      if (addend && g.N % 4 == 0 && ld % 4 == 0 && (uintptr_t)addend % 16 == 0 && (int64_t)g.M * ld < (1 << 29)) {   // uniform
        added = true;
        const __amdgpu_buffer_rsrc_t rsD = make_rsrc(addend, (uint32_t)(((int64_t)(g.M - 1) * ld + g.N) * 4));
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const int m = m0 + wm0 + 16 * i + r;
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            const int c = 32 * (j / 2) + 4 * (j % 2);
            const uint32_t at = m < g.M && c < cols ? (uint32_t)((m * ld + n + c) * 4) : kOobOffset;
            add[i][j] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rsD, at, 0, 0));
          }
        }
      }
    }
  };
  if constexpr (EARLY_ADD) {
    if (g.c_dtype == MX_F32 && g.k_splits <= 1) load_addend();
    __builtin_amdgcn_sched_barrier(0);
  }

  // ---- prologue ---------------------------------------------------------------------------------------------------------
  if constexpr (ANY) load_any(q0);
#pragma unroll
  for (int k = 0; k < NS; ++k) {
    if (!ANY && Sched::prologue_scales(k)) load_scales(q0 + k / SPQ);
    issue(s0 + k, k, 0, 1);
    __builtin_amdgcn_sched_barrier(0);   // the waits count on this order
  }
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(ANY ? Sched::any_prologue_wait() : Sched::prologue_wait()));
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (ANY) {
    store_any(q0);
    load_any(q0 + 1);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  read_scales(q0);
  {
    using Z = std::integral_constant<int, 0>;
#pragma unroll
    for (int j = 0; j < NT; ++j) read_b(0, Z{}, j);
#pragma unroll
    for (int i = 0; i < MT; ++i) read_a(0, Z{}, i);
  }
  take_scales();

  int buf = 0;                        // buffer of stage s
  auto stage = [&](int Q, auto tc) {
    constexpr int t = decltype(tc)::value, set = t & 1;
    using Nx = std::integral_constant<int, set ^ 1>;
    const int s = Q * SPQ + t;
    if (s >= s1) return;              // uniform
    // stage s + 1 (requested NS - 1 iterations ago) has landed; younger are NS - 2 stages and the scales requested since
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(ANY ? Sched::any_stage_wait() : Sched::stage_wait(t)));
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (t == 0) {
      if constexpr (ANY) {
        store_any(Q + 1);             // requested a quad ago; the slot was last read two quads ago
        load_any(Q + 2);
      } else {
        load_scales(Q + SD);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!SPREAD) {
      issue(s + NS, buf, 0, 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    const int nbuf = buf + 1 == NS ? 0 : buf + 1;
    // the next quad's scales landed before this iteration's barrier (they were requested ahead of stage s + 1)
    if constexpr (t == SPQ - 1) read_scales(Q + 1);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      read_b(nbuf, Nx{}, i);
      read_a(nbuf, Nx{}, i);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) {
        const int u = t * KS + kk;    // K-step of the quad
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = mfma_scaled<C::BF, C::AF>(bf[set][kk][j], af[set][kk][i], acc[i][j], BP ? u : j, BP ? sb[j] : sb[u],
                                                AP ? u : i, AP ? sa[i] : sa[u]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (SPREAD) {
        issue(s + NS, buf, i, MT);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    buf = nbuf;
  };
  for (int Q = q0; Q < q1; ++Q) {
    stage(Q, std::integral_constant<int, 0>{});
    stage(Q, std::integral_constant<int, 1>{});
    if constexpr (SPQ == 4) {
      stage(Q, std::integral_constant<int, 2>{});
      stage(Q, std::integral_constant<int, 3>{});
    }
    take_scales();
  }

  // ---- epilogue: lane (r, gq) of tile pair (2 jp, 2 jp + 1) holds row 16 i + r, columns 32 jp + 8 gq .. + 7 -------------
  auto store = [&](auto kind) {        // 0: fp32, 1: bf16, 2: fp32 partial product of a split
    constexpr int kd = decltype(kind)::value;
    using OutT = std::conditional_t<kd == 1, uint16_t, float>;
    OutT* const Cp = kd == 2 ? (OutT*)(g.partial + (int64_t)split * g.M * g.N) : (OutT*)g.C + (int64_t)bz * g.c_batch;
    const int64_t ld = kd == 2 ? g.N : g.ldc;
    if constexpr (kd == 0 && !GROUPED && !EARLY_ADD) load_addend();
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int m = m0 + wm0 + 16 * i + r;
      int64_t row = m;
      bool ok = m < g.M;
      float w = 1.f;
      if constexpr (GROUPED) {
        const int id = ok ? g.sorted_token_ids[m] : 0x7FFFFFFF;
        ok = ok && id >= 0 && id < g.num_valid_ids;
        row = id;
        if (ok && g.topk_weights) w = g.topk_weights[id];
      }
      if (!ok) continue;
#pragma unroll
      for (int jp = 0; jp < NT / 2; ++jp) {
        v4f v0 = acc[i][2 * jp], v1 = acc[i][2 * jp + 1];
        if constexpr (GROUPED) { v0 *= w; v1 *= w; }
        const int64_t off = row * ld + n + 32 * jp;
        if (kd == 0 && added) {
          if constexpr (kd == 0 && !GROUPED) { v0 += add[i][2 * jp]; v1 += add[i][2 * jp + 1]; }
        } else if (kd != 2 && g.acc) add8_edge<float>(g.acc + (int64_t)bz * g.c_batch + off, v0, v1, cols - 32 * jp);
        else if (kd != 2 && g.accumulate) add8_edge<OutT>(Cp + off, v0, v1, cols - 32 * jp);
        store8_edge<OutT>(Cp + off, v0, v1, cols - 32 * jp);
      }
    }
  };
  if (g.k_splits > 1) store(std::integral_constant<int, 2>{});
  else if (g.c_dtype == MX_F32) store(std::integral_constant<int, 0>{});
  else store(std::integral_constant<int, 1>{});
}

template <class C, int NS, int AS, int BS, bool GROUPED, bool SPREAD>
__global__ __launch_bounds__(256, NS == 2 || (C::BM == 64 && NS == 4) ? 2 : 1) void t128_kernel(const T128Args g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem_generic[];
  t128_tile<C, NS, AS, BS, GROUPED, SPREAD>(g, (lds_u8*)smem_generic, blockIdx.x, blockIdx.y, blockIdx.z);
  __builtin_amdgcn_s_waitcnt(0x0F70);   // the trailing zero-fill DMA has left the queue before the LDS is given back
}

// ---- list of problems: persistent workgroups walk the concatenated tile list -------------------------------------------
constexpr int kListMax = 32;
struct ListProblem {
  const uint8_t* A; const uint8_t* B; const uint8_t* As; const uint8_t* Bs; void* C;
  int64_t lda, ldb, ldas, ldbs, ldc;
  int32_t M, N, K;
  int16_t c_dtype, scales;             // kScale... of both operands
};
struct T128List {
  ListProblem p[kListMax];
  int32_t first_tile[kListMax + 1];
  int32_t n;
};

// Problems whose scales are read in place and problems whose scales were re-laid share the launch: one after the other, two
// launches of 24 problems of 96 .. 1536 took 16.6 + 10.9 us, each waiting for its own longest product.
template <class C>
__global__ __launch_bounds__(256, 2) void t128_list_kernel(const T128List gl) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem_generic[];
  lds_u8* const smem = (lds_u8*)smem_generic;
  const int total = gl.first_tile[gl.n];
  for (int t = blockIdx.x; t < total; t += gridDim.x) {   // uniform per workgroup
    int i = 0;
    while (i + 1 < gl.n && t >= gl.first_tile[i + 1]) ++i;
    const ListProblem& q = gl.p[i];
    T128Args g = {};
    g.A = q.A; g.B = q.B; g.As = q.As; g.Bs = q.Bs; g.C = q.C;
    g.lda = q.lda; g.ldb = q.ldb; g.ldas = q.ldas; g.ldbs = q.ldbs; g.ldc = q.ldc;
    g.M = q.M; g.N = q.N; g.K = q.K; g.c_dtype = q.c_dtype;
    g.k_splits = 1;
#if defined(__HIP_DEVICE_COMPILE__)   // (the host pass, which needs the kernel's stub only, refuses the call)
    if (q.scales == kScalePlain) t128_tile<C, 2, kScalePlain, kScalePlain, false>(g, smem, t - gl.first_tile[i], 0, 0);
    else if (q.scales == kScaleAny) t128_tile<C, 2, kScaleAny, kScaleAny, false>(g, smem, t - gl.first_tile[i], 0, 0);
    else t128_tile<C, 2, kScaleNative, kScaleNative, false>(g, smem, t - gl.first_tile[i], 0, 0);
#endif
    // the tile's trailing (zero-fill) DMA has left the queue and every wave is done with the LDS stages before
    // the next tile's loads reuse them
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
  }
}

template <class C, int NS, int AS, int BS, bool GROUPED, bool SPREAD = kSpread<C, NS, AS>>
int launch_one(const T128Args& g, hipStream_t stream) {
  auto kern = t128_kernel<C, NS, AS, BS, GROUPED, SPREAD>;
  constexpr int lds = NS * C::STAGE + ((NS + 4 / C::KSUB - 1) / (4 / C::KSUB) + 1) * 4096;
  static int attr_done = 0;   // benign race: the attribute call is idempotent
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "hipFuncSetAttribute(%d bytes LDS): %s", lds, hipGetErrorString(e));
    attr_done = 1;
  }
  const int64_t tiles = (int64_t)((g.M + C::BM - 1) / C::BM) * ((g.N + C::BN - 1) / C::BN);
  if (tiles <= 0) return MX_OK;
  hipError_t e = launch_kernel(kern, dim3((unsigned)tiles, (unsigned)g.k_splits, (unsigned)g.batch), dim3(256), lds, stream, g);
  if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "t128_kernel launch: %s", hipGetErrorString(e));
  return MX_OK;
}

template <class C>
int launch_list(const T128List& gl, hipStream_t stream) {
  auto kern = t128_list_kernel<C>;
  constexpr int lds = 2 * C::STAGE + 2 * 4096;
  static int attr_done = 0;   // benign race: the attribute call is idempotent
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "hipFuncSetAttribute(%d bytes LDS): %s", lds, hipGetErrorString(e));
    attr_done = 1;
  }
  const int total = gl.first_tile[gl.n];
  if (total <= 0) return MX_OK;
  hipError_t e = launch_kernel(kern, dim3((unsigned)(total < 512 ? total : 512)), dim3(256), lds, stream, gl);   // two per CU
  if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "t128_list_kernel launch: %s", hipGetErrorString(e));
  return MX_OK;
}

}  // namespace

// One element-format pair per compilation of this file (T128_PAIR), so that the pairs build in parallel.
template <int AF, int BF>
int t128_pair(const T128Args& g, hipStream_t stream) {
  using C = Cfg<AF, BF, 128, 128, 2, 2>;
  if (g.sorted_token_ids)
    return g.a_plain ? launch_one<C, 2, kScalePlain, kScaleNative, true>(g, stream)
                     : launch_one<C, 2, kScaleNative, kScaleNative, true>(g, stream);
  // (A packed with B plain does not occur: the entry points re-lay B first)
  const int64_t wgs = (int64_t)((g.M + 127) / 128) * ((g.N + 127) / 128) * g.k_splits * g.batch;
  auto depth = [&](auto cfg, auto ns) {
    using D = decltype(cfg);
    constexpr int NS = decltype(ns)::value;
    if (g.a_plain == kT128ScalesAny) {
      if constexpr (D::BM == 64 && NS == 8)
        if (!t128_any_spread(g.K, g.k_splits, D::KSUB)) return launch_one<D, NS, kScaleAny, kScaleAny, false, false>(g, stream);
      return launch_one<D, NS, kScaleAny, kScaleAny, false>(g, stream);
    }
    return !g.a_plain   ? launch_one<D, NS, kScaleNative, kScaleNative, false>(g, stream)
           : !g.b_plain ? launch_one<D, NS, kScalePlain, kScaleNative, false>(g, stream)
                        : launch_one<D, NS, kScalePlain, kScalePlain, false>(g, stream);
  };
  const int64_t small = t128_small_tiles(g.M, g.N) * g.k_splits * g.batch;
  if (small <= kT128SmallTiles) {
    using S = Cfg<AF, BF, 64, 64, 2, 2>;
    return small <= 256 ? depth(S{}, std::integral_constant<int, 8>{}) : depth(S{}, std::integral_constant<int, 4>{});
  }
  return wgs <= 256 ? depth(C{}, std::integral_constant<int, 4>{}) : depth(C{}, std::integral_constant<int, 2>{});
}
template <int AF, int BF>
int t128_list_pair(const T128Args* problems, int n, hipStream_t stream) {
  using C = Cfg<AF, BF, 128, 128, 2, 2>;
  for (int i0 = 0; i0 < n; i0 += kListMax) {
    T128List gl = {};
    int64_t total = 0;
    for (int i = i0; i < n && i < i0 + kListMax; ++i) {
      const T128Args& g = problems[i];
      ListProblem& q = gl.p[gl.n];
      q.A = g.A; q.B = g.B; q.As = g.As; q.Bs = g.Bs; q.C = g.C;
      q.lda = g.lda; q.ldb = g.ldb; q.ldas = g.ldas; q.ldbs = g.ldbs; q.ldc = g.ldc;
      q.M = g.M; q.N = g.N; q.K = g.K; q.c_dtype = (int16_t)g.c_dtype; q.scales = (int16_t)(g.a_plain && g.b_plain ? g.a_plain : kScaleNative);
      gl.first_tile[gl.n] = (int32_t)total;
      total += (int64_t)((g.M + 127) / 128) * ((g.N + 127) / 128);
      if (total > 0x7FFFFFFF) return set_error(MX_ERR_SHAPE, "gemm list: too many tiles");
      ++gl.n;
    }
    gl.first_tile[gl.n] = (int32_t)total;
    if (int rc = launch_list<C>(gl, stream)) return rc;
  }
  return MX_OK;
}

#define T128_INSTANCES(AF, BF)                                             \
  template int t128_pair<AF, BF>(const T128Args&, hipStream_t);            \
  template int t128_list_pair<AF, BF>(const T128Args*, int, hipStream_t);
#if T128_PAIR == 1
T128_INSTANCES(MX_E5M2, MX_E5M2)
#elif T128_PAIR == 2
T128_INSTANCES(MX_E2M1, MX_E2M1)
#elif T128_PAIR == 3
T128_INSTANCES(MX_E4M3, MX_E2M1)
#else
T128_INSTANCES(MX_E4M3, MX_E4M3)
#define T128_EXTERN(AF, BF)                                                \
  extern template int t128_pair<AF, BF>(const T128Args&, hipStream_t);     \
  extern template int t128_list_pair<AF, BF>(const T128Args*, int, hipStream_t);
T128_EXTERN(MX_E5M2, MX_E5M2)
T128_EXTERN(MX_E2M1, MX_E2M1)
T128_EXTERN(MX_E4M3, MX_E2M1)

int launch_gemm_t128(const T128Args& g, hipStream_t stream) {
#define MX_CASE(AF, BF) \
  if (g.a_fmt == AF && g.b_fmt == BF) return t128_pair<AF, BF>(g, stream);
  MX_CASE(MX_E4M3, MX_E4M3)
  MX_CASE(MX_E5M2, MX_E5M2)
  MX_CASE(MX_E2M1, MX_E2M1)
  MX_CASE(MX_E4M3, MX_E2M1)
#undef MX_CASE
  return set_error(MX_ERR_DTYPE, "MFMA kernel: unsupported element format pair (%d, %d)", g.a_fmt, g.b_fmt);
}

int launch_gemm_t128_list(const T128Args* p, int n, hipStream_t stream) {
  for (int i = 0; i < n; ++i)
    if (p[i].a_fmt != p[0].a_fmt || p[i].b_fmt != p[0].b_fmt || !p[i].a_plain != !p[i].b_plain)
      return set_error(MX_ERR_INVALID, "gemm list: problems of one launch must share formats, their operands the scale layout");
#define MX_CASE(AF, BF) \
  if (p[0].a_fmt == AF && p[0].b_fmt == BF) return t128_list_pair<AF, BF>(p, n, stream);
  MX_CASE(MX_E4M3, MX_E4M3)
  MX_CASE(MX_E5M2, MX_E5M2)
  MX_CASE(MX_E2M1, MX_E2M1)
  MX_CASE(MX_E4M3, MX_E2M1)
#undef MX_CASE
  return set_error(MX_ERR_DTYPE, "gemm list: unsupported element format pair (%d, %d)", p[0].a_fmt, p[0].b_fmt);
}
#endif

}  // namespace mx
