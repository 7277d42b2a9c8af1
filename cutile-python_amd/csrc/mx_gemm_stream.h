// Weight-streaming block-scaled GEMM for few rows of X (decode): C[M, N] (+)= X[M, K] (8-bit MX) x W[N, K]^T with 8-bit
// or FP4 weights; the body shared by the plain and the mixture-of-experts launches.
//
// Bound: reading W once from HBM.  Every wave works on its own: it streams NT 16-row tiles of W over its own range of
// K into registers and the matching columns of X through its own corner of LDS, multiplies, and meets the other waves
// of its workgroup only once, when the partial sums of the K ranges are added in LDS.  No barrier in the stream and
// nothing shared, so the waves of a CU drift apart and keep its memory queue full.
//   * W: 8 rows x 128 bytes per load instruction, re-sorted into the MFMA operand layout by a write to and a read from a
//     4 KiB scratch area of the wave in LDS (LDS serves a wave in order: no wait between the two).  Loading the operand
//     layout directly (16 rows x 16 bytes per lane group) costs the address unit one request per lane instead of one per
//     four: a bare stream of 117 MB with as many bytes of X beside it takes 33.5 us that way and 25.5 us this way (23 us
//     without X).
//   * X: one K-step of MT 16-row tiles is 2 MT KiB; it comes by LDS-DMA, also 8 rows x 128 bytes per instruction.  16-byte
//     chunks are XOR-swizzled by row: conflict-free fragment reads.
//   * a stage is 128 bytes of a row of W: one K-step of 128 elements, two for FP4 weights.  Two stages are in the queue;
//     four measured no faster at any size, and the memory pipe returns data in request order, so X cannot run on a
//     shorter leash than W.
//   * scales of W: the native layout (one 16-byte load per lane is a 64-row group's scales for a K-quad of four
//     K-steps, the tile picked by the instruction's byte select) or plain [N, K/32] rows (16 bytes of a row per quad, the
//     lane's byte shifted down); X: plain rows.
#pragma once

#include <type_traits>

#include "mx_gemm_pp.h"   // vmcnt_imm
#include "mx_gemm_tile.h"
#include "mx_load_once.h"
#include "mx_stream.h"

namespace mx {

// UP: the four tiles of a wave are 32 rows of the gate half of W and the 32 rows of the up half that belong to them.
// ONCE: W is read non-temporally (stream_loads_once).
template <int XF_, int WF_, int NT_, int MT_, bool PACKED_, int WAVES_ = 8, bool UP_ = false, bool ONCE_ = false>
struct StreamCfg {
  static constexpr int XF = XF_, WF = WF_, NT = NT_, MT = MT_, WAVES = WAVES_;
  static constexpr bool PACKED = PACKED_, UP = UP_;
  static constexpr int NSW = PACKED ? (UP ? 2 : 1) : NT;  // scale registers (x 4) of W per K-quad
  static constexpr int SK = WF == MX_E2M1 ? 2 : 1;        // K-steps per stage
  static constexpr int SPQ = 4 / SK;                      // stages per K-quad
  static constexpr int WEB = WF == MX_E2M1 ? 4 : 8;
  static constexpr int L = 2 * MT * SK + 2 * NT;          // load instructions per stage
  // For units of whole 64-row groups: 8 experts of 4096 x 14336, 12 rows each, up + down projection FP8 257 -> 226 us (5.7 -> 6.4
  // TB/s), FP4 149 -> 136; 28672 x 8192 FP8, 16 rows 45.2 -> 40.9.  Narrow units (one or two tiles, which split K over more
  // waves) gain nothing, and 4096 x 14336 FP8 at 24 rows loses: 18.1 -> 19.9.  (Instances of their own: both kinds of load in
  // one kernel cost small layers 5 % in instruction fetches.)
  static constexpr int W_POLICY = ONCE_ ? kLoadOnce : 0;
  static_assert(!ONCE_ || NT == 4, "");
  static constexpr int NSC = MT + NSW;      // scale load instructions per K-quad
  static constexpr int XSLOT = MT * SK * 2048;            // LDS bytes of one stage of X
  // tiles of W re-sorted at a time (one where that lets two workgroups of four waves share a CU's LDS)
  static constexpr int TP = NT >= 2 && !(WAVES == 4 && XSLOT == 8192) ? 2 : 1;
  static constexpr int WAVE_BYTES = 2 * XSLOT + TP * 2048;
  static constexpr int RED = WAVES * NT * MT * 1024;   // partial sums: [wave][tile][lane] float4
  static constexpr int LDS_BYTES = WAVES * WAVE_BYTES > RED ? WAVES * WAVE_BYTES : RED;
  static_assert(!UP || NT == 4, "two tiles of gate, two of up");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");
  static_assert(L + NSC < 63, "vmcnt range");
};

// What one wave multiplies: descriptors of its operands.
struct StreamWave {
  __amdgpu_buffer_rsrc_t rsX, rsXs, rsW, rsWs;
};

// Row of a DMA / load instruction's lane (8 rows x 128 bytes) and the 16-byte chunk of the row that it fetches: X goes to
// LDS as it comes, so its chunks are swizzled on the way in; W is swizzled when it is written to the scratch area.
__device__ inline uint32_t stream_x_col(int q, int lane) { return (uint32_t)(((lane & 7) ^ swz<8>(8 * q + (lane >> 3))) << 4); }

// acc[i][j] of the wave: rows 16 i + lane % 16 of X, tile j0[0] + j of its group of W, K-quads [Q0, Q1) (the last one may be
// partial: ksteps in all).  xvo: lane offsets of the 2 MT DMA instructions of a K-step of X (kOobOffset: no such row);
// xso: lane offset of the 16 scale bytes of row 16 i + lane % 16; wvo: lane offsets of the 2 NT load instructions of a
// stage of W (rows 8 h + lane / 8 of tile j in instruction 2 j + h); wso: lane offset of the scales of tile j's row
// lane % 16 (packed: one, of the group; UP: two, of the groups that the gate and the up rows lie in, whose first tiles
// are j0[0] and j0[1]).
template <class C>
__device__ __forceinline__ void stream_products(const StreamWave& w, lds_u8* const lds, const uint32_t (&xvo)[2 * C::MT],
                                                const uint32_t (&xso)[C::MT], const uint32_t (&wvo)[2 * C::NT],
                                                const uint32_t (&wso)[C::NSW], const int (&j0)[C::UP ? 2 : 1], const int Q0,
                                                const int Q1, const int ksteps, v4f (&acc)[C::MT][C::NT]) {
  constexpr int NT = C::NT, MT = C::MT, SK = C::SK, TP = C::TP;
  typedef __attribute__((address_space(3))) v4i lds_w4i;
  const int lane = threadIdx.x & 63, r = lane & 15, gq = lane >> 4;
  const int s1 = Q1 * 4 < ksteps ? Q1 * 4 : ksteps;
  lds_u8* const scr = lds + 2 * C::XSLOT;
  v4i wr[2][NT][2];
  v4i sx[MT], sxn[MT], sw[C::NSW], swn[C::NSW];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};

  auto load_scales = [&](int Q, v4i (&x)[MT], v4i (&ws)[C::NSW]) {
    const bool live = Q < Q1;
#pragma unroll
    for (int i = 0; i < MT; ++i)
      x[i] = __builtin_amdgcn_raw_buffer_load_b128(w.rsXs, live ? xso[i] : kOobOffset, Q * 16, 0);
    if constexpr (C::PACKED) {
#pragma unroll
      for (int j = 0; j < C::NSW; ++j)
        ws[j] = __builtin_amdgcn_raw_buffer_load_b128(w.rsWs, live ? wso[j] : kOobOffset, Q * 1024, 0);
    } else {
#pragma unroll
      for (int j = 0; j < NT; ++j)
        ws[j] = __builtin_amdgcn_raw_buffer_load_b128(w.rsWs, live ? wso[j] : kOobOffset, Q * 16, 0);
    }
  };
  // stage p (K-steps SK p ...) into ring slot `slot`; K-steps at or beyond s1 fetch nothing
  auto issue = [&](int p, auto slotc) {
    constexpr int slot = decltype(slotc)::value;
#pragma unroll
    for (int kk = 0; kk < SK; ++kk) {
      const int s = p * SK + kk;
#pragma unroll
      for (int q = 0; q < 2 * MT; ++q)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(w.rsX, (lds_void*)(lds + slot * C::XSLOT + (kk * 2 * MT + q) * 1024), 16,
                                                 s < s1 ? xvo[q] : kOobOffset, s * 128, 0, 0);
    }
    const bool live = p * SK < s1;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        wr[slot][j][h] = __builtin_amdgcn_raw_buffer_load_b128(w.rsW, live ? wvo[2 * j + h] : kOobOffset, p * 128, C::W_POLICY);
    __builtin_amdgcn_sched_barrier(0);
  };
  load_scales(Q0, sx, sw);
  __builtin_amdgcn_sched_barrier(0);
  issue(Q0 * C::SPQ, std::integral_constant<int, 0>{});
  issue(Q0 * C::SPQ + 1, std::integral_constant<int, 1>{});
  const int swx = swz<8>(r);
  // where lane's chunk of load instruction h of a tile goes: row 8 h + lane / 8, chunk lane % 8
  const int wpos = (lane >> 3) * 128 + (((lane & 7) ^ swz<8>(lane >> 3)) << 4);
  const int wpos1 = (8 + (lane >> 3)) * 128 + (((lane & 7) ^ swz<8>(8 + (lane >> 3))) << 4);
  auto stage = [&](int Q, auto tc) {
    constexpr int t = decltype(tc)::value, slot = t % 2;
    const int p = Q * C::SPQ + t;
    // everything of this stage has arrived; younger are the next stage and, if this stage was requested in the quad
    // before, the scales of the next quad
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(C::L + (t < 2 ? C::NSC : 0)));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (p * SK < s1) {   // uniform
      v8i xf[SK][MT];
#pragma unroll
      for (int kk = 0; kk < SK; ++kk)
#pragma unroll
        for (int i = 0; i < MT; ++i) xf[kk][i] = load_frag<128, 8>(lds + slot * C::XSLOT + kk * MT * 2048, 16 * i + r, 0, gq, swx);
#pragma unroll
      for (int jb = 0; jb < NT; jb += TP) {
#pragma unroll
        for (int j = jb; j < jb + TP; ++j) {
          *(lds_w4i*)(scr + (j - jb) * 2048 + wpos) = wr[slot][j][0];
          *(lds_w4i*)(scr + (j - jb) * 2048 + wpos1) = wr[slot][j][1];
        }
        v8i wf[SK][TP];
#pragma unroll
        for (int kk = 0; kk < SK; ++kk)
#pragma unroll
          for (int j = 0; j < TP; ++j) wf[kk][j] = load_frag<128, C::WEB>(scr + j * 2048, r, kk, gq, swx);
#pragma unroll
        for (int kk = 0; kk < SK; ++kk) {
          constexpr int u0 = t * SK;
          const int u = u0 + kk;         // K-step of the quad
          if (kk > 0 && p * SK + kk >= s1) continue;   // uniform
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            const int xs = (int)((uint32_t)sx[i][u] >> (8 * gq));
#pragma unroll
            for (int j = jb; j < jb + TP; ++j) {
              if constexpr (C::PACKED) {
                // a full group's tiles are the four bytes; fewer tiles of a group start at byte j0, shifted down
                constexpr bool whole = NT == 4 && !C::UP;
                const int g = C::UP ? j / 2 : 0;
                const int ws = whole ? sw[0][u] : (int)((uint32_t)sw[g][u] >> (8 * j0[g]));
                acc[i][j] = mfma_scaled<C::WF, C::XF>(wf[kk][j - jb], xf[kk][i], acc[i][j], C::UP ? j % 2 : j, ws, 0, xs);
              } else {
                acc[i][j] = mfma_scaled<C::WF, C::XF>(wf[kk][j - jb], xf[kk][i], acc[i][j], 0,
                                                      (int)((uint32_t)sw[j][u] >> (8 * gq)), 0, xs);
              }
            }
          }
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the fragments are out of the slot that is refilled now
    __builtin_amdgcn_sched_barrier(0);
    issue(p + 2, std::integral_constant<int, slot>{});
  };
  for (int Q = Q0; Q < Q1; ++Q) {
    load_scales(Q + 1, sxn, swn);
    __builtin_amdgcn_sched_barrier(0);
    stage(Q, std::integral_constant<int, 0>{});
    stage(Q, std::integral_constant<int, 1>{});
    if constexpr (C::SPQ == 4) {
      stage(Q, std::integral_constant<int, 2>{});
      stage(Q, std::integral_constant<int, 3>{});
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) sx[i] = sxn[i];
#pragma unroll
    for (int j = 0; j < C::NSW; ++j) sw[j] = swn[j];
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // the trailing zero-fill DMA has left the queue: LDS may be reused
}

}  // namespace mx
