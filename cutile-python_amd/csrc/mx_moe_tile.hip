// Mixture-of-experts layer at medium sizes: experts of some 24 to 128 rows (which layers: moe_plan in mx_api.hip).
//
// Bound: reading the experts' weights once.  Streaming them past every few rows (mx_moe.hip) reads them again for each 32 rows;
// the grouped 256 x 256 kernel has one workgroup per CU, whose two stages in flight ask for 4 TB/s of them, and needs slot
// arrays, re-laid scales, a bf16 activation written and read and a launch that adds up the split last round around it.  Here:
//   moe_tiles_kernel:       the routed copies of every expert, in tiles of 64 (FP4 and long rows of W: 128, moe_tile_rows);
//   moe_tile_kernel<UP>:    a tile x (64 gate + 64 up columns), SiLU(gate) * up and its MX quantisation in the epilogue;
//   moe_tile_kernel<DOWN>:  a tile x 128 columns, fp32, K in several ranges where there would be too few workgroups;
//   moe_combine_kernel:     adds up the ranges and a token's copies (mx_moe.hip).
// A workgroup is four waves of 32 x 64 (64 x 64) on the schedule of the 128 x 128 kernel (order of the requests and counted waits:
// mx_t128_schedule.h): 80 KiB of LDS, two workgroups on a CU, so that one's start and output lie behind the other's stream and
// together they have up to six stages of 16 KiB of weights in flight.  (Eight waves on 128 or 256 rows, one workgroup per CU and
// four or three stages deep, leave start and output open: 8 experts of 2048 x 7168, 32 and 64 rows each, FP8 93 | 112 | 147 and
// 114 | 118 | 153 us.)
// us per layer before (streamed or 256-row tiles) -> now: 8 experts of 4096 x 14336, 40 rows each FP8 368 -> 274, FP4 257 -> 177; 8 of
// 2048 x 7168, 75 rows 164 -> 117, 134 -> 95; 16 of 3072 x 4096, 64 rows 202 -> 170, 152 -> 125; 64 of 2048 x 1024, 38 rows 173 -> 104,
// 137 -> 79.  The first reads 1.41 GB at 5.3 TB/s, where a bare stream of them in these pieces reaches 5.8 (6.5 non-temporally).
#include <type_traits>

#include "mx_gemm_pp.h"      // vmcnt_imm
#include "mx_gemm_tile.h"
#include "mx_load_once.h"
#include "mx_moe_tile.h"
#include "mx_quant.h"
#include "mx_t128_schedule.h"

namespace mx {
namespace {

// ---- routed copies -> row tiles ------------------------------------------------------------------------------------------
// One workgroup: up to 16 ids per thread stay in registers, an LDS counter per expert hands out the places (the order of an
// expert's copies is not fixed; every copy's result is its own).
constexpr int kTilesThreads = 1024, kTilesPer = kMoeTileMaxIds / kTilesThreads;
__global__ __launch_bounds__(kTilesThreads) void moe_tiles_kernel(const int32_t* __restrict__ ids, int id_shift, int n, int E,
                                                                  int tile_rows, MoeTile* __restrict__ tiles,
                                                                  int32_t* __restrict__ slots, int max_tiles) {
  __shared__ int32_t count[kMoeTileMaxExperts], first[kMoeTileMaxExperts], wave_sum[kTilesThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int e[kTilesPer], place[kTilesPer];
#pragma unroll
  for (int k = 0; k < kTilesPer; ++k) {
    const int i = k * kTilesThreads + tid;
    e[k] = i < n ? ids[(int64_t)i << id_shift] : -1;
    if (e[k] >= E) e[k] = -1;
  }
  count[tid] = 0;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kTilesPer; ++k)
    if (e[k] >= 0) place[k] = atomicAdd(&count[e[k]], 1);
  __syncthreads();
  // first tile of every expert: thread = expert
  const int mine = count[tid], t = (mine + tile_rows - 1) / tile_rows;
  int sum = t;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(sum, d);
    if (lane >= d) sum += o;
  }
  if (lane == 63) wave_sum[wave] = sum;
  __syncthreads();
  int before = 0, total = 0;
#pragma unroll
  for (int w = 0; w < kTilesThreads / 64; ++w) {
    if (w < wave) before += wave_sum[w];
    total += wave_sum[w];
  }
  const int run = before + sum - t;
  first[tid] = run;
  for (int i = 0; i < t; ++i) tiles[run + i] = MoeTile{tid, mine - i * tile_rows, run, t};
  for (int i = total + tid; i < max_tiles; i += kTilesThreads) tiles[i] = MoeTile{0, 0, 0, 1};
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kTilesPer; ++k)
    if (e[k] >= 0) slots[first[e[k]] * tile_rows + place[k]] = k * kTilesThreads + tid;
}

// ---- the products ----------------------------------------------------------------------------------------------------------
// A stage is KS K-steps of 128 elements.  Plain loads of FP4 weights take 64 bytes of a row at a time and have four stages in flight;
// non-temporal ones take whole lines, two K-steps (X's then lie one behind the other), as a line's second half would come from memory
// again (a bare stream in pieces of 64 bytes: 5.5 TB/s plain, 4.4 non-temporal, of 128 bytes 5.8 and 6.4).
template <int WF_, bool UP_, int BM_, bool ONCE_, int NS_, int KS_>
struct MoeTileCfg {
  static constexpr int WF = WF_, NS = NS_, BM = BM_, BN = kMoeTileCols, KS = KS_, SPQ = 4 / KS;
  static constexpr bool UP = UP_, ONCE = ONCE_;
  static constexpr int W_EB = WF == MX_E2M1 ? 4 : 8, MT = BM / 32, NT = 4;   // waves: 2 x 2 of BM / 2 rows x 64 columns
  static constexpr int RB = 16 * W_EB * KS, CPR = RB / 16, RPI = 64 / CPR;   // bytes, 16-byte chunks of a row of W, rows per load
  static constexpr int A_STEP = BM * 128, A_STAGE = KS * A_STEP, STAGE = A_STAGE + BN * RB;
  static constexpr int AL = BM / 32, BL = BN / RPI / 4, TL = KS * AL + BL;   // loads per wave: of a K-step of X, of W, of a stage
  static constexpr int LDS = NS * STAGE + (T128Schedule<NS, SPQ, TL>::SD + 1) * 4096;
  static_assert(LDS <= 80 * 1024, "two workgroups per CU");
};

template <class C>
__global__ __launch_bounds__(256, 2) void moe_tile_kernel(const MoeTileArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)   // (the host pass, which needs the kernel's stub only, refuses lambdas around these builtins)
  constexpr int NS = C::NS, MT = C::MT, NT = C::NT, KS = C::KS, SPQ = C::SPQ;
  constexpr bool UP = C::UP;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem_generic[];
  lds_u8* const smem = (lds_u8*)smem_generic;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, gq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  // ---- tile: XCD x (workgroup ids are dealt round-robin) has the column tiles (and K ranges) v = x, x + 8, ... of all rows.
  // Row by row, and the row tiles of one expert next to each other, so that they meet on their weights in the XCD's L2.
  const int cols = UP ? a.F / 64 : (a.N + 127) / 128, v_all = cols * a.splits, per = (v_all + 7) >> 3;
  const int loc = blockIdx.x >> 3;
  MoeTile tile = a.tiles[loc / per];
  const int expert = __builtin_amdgcn_readfirstlane(tile.expert), run = __builtin_amdgcn_readfirstlane(tile.run);
  const int run_tiles = __builtin_amdgcn_readfirstlane(tile.run_tiles);
  int rows = __builtin_amdgcn_readfirstlane(tile.rows);
  if (rows == 0) return;                             // uniform: a tile that this routing has no use for
  const int in = loc - run * per, tr = in % run_tiles, v = in / run_tiles * 8 + (blockIdx.x & 7);
  if (v >= v_all) return;
  rows += (loc / per - run - tr) * C::BM;     // of the expert from row tile run + tr on
  const int split = v / cols, col = v - split * cols;
  const int32_t* const slots = a.slots + (int64_t)(run + tr) * C::BM;

  const int KQ = (a.K + 511) / 512, q0 = split * KQ / a.splits, q1 = (split + 1) * KQ / a.splits;
  const int nst = (a.K / 128 + KS - 1) / KS, s0 = q0 * SPQ, s1 = q1 * SPQ < nst ? q1 * SPQ : nst;   // stages [s0, s1)

  const __amdgpu_buffer_rsrc_t rsA = make_rsrc(a.X, operand_bytes(a.x_rows, a.ldx, a.K));
  const __amdgpu_buffer_rsrc_t rsB = make_rsrc(a.W + (int64_t)expert * a.w_es, operand_bytes(a.N, a.ldw, (int64_t)a.K * C::W_EB / 8));
  const __amdgpu_buffer_rsrc_t rsAs = make_rsrc(a.Xs, operand_bytes(a.x_rows, a.ldxs, a.K / 32));
  const __amdgpu_buffer_rsrc_t rsBs = make_rsrc(a.Ws + (int64_t)expert * a.ws_es, (uint32_t)(packed_scale_dwords(a.N, a.K) * 4));

  // ---- DMA: instruction q of wave w fills 1 KiB of the stage: rows RPI * (4 q + w) ... -----------------------------------------
  constexpr int AL = C::AL, BL = C::BL;
  uint32_t avo[AL], bvo[BL];
  const int a_lr = 8 * wave + (lane >> 3), b_lr = C::RPI * wave + lane / C::CPR;   // row of instruction 0
  const int a_col = ((lane & 7) ^ swz<8>(a_lr)) * 16, b_col = ((lane % C::CPR) ^ swz_bperm<C::CPR>(b_lr)) * 16;
#pragma unroll
  for (int q = 0; q < AL; ++q) {
    const int row = 32 * q + a_lr;
    avo[q] = kOobOffset;
    if (row < rows) avo[q] = (uint32_t)(slots[row] / a.replicas * a.ldx + a_col);
  }
#pragma unroll
  for (int q = 0; q < BL; ++q) {
    const int row = 4 * C::RPI * q + b_lr;            // of the stage; the up projection's rows 64 .. 127 are the up half's
    const int n = UP ? (row >> 6) * a.F + 64 * col + (row & 63) : 128 * col + row;
    bvo[q] = n < a.N ? (uint32_t)(n * a.ldw + b_col) : kOobOffset;
  }
  const int Kb = a.K * C::W_EB / 8;                  // bytes of a row of W
  auto issue = [&](int s, int buf) {                 // (a K-step at or beyond the end arrives as zeros)
    lds_u8* const base = smem + buf * C::STAGE + wave * 1024;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      const bool in_k = s < s1 && (KS == 1 || (s * KS + kk) * 128 < a.K);   // uniform
#pragma unroll
      for (int q = 0; q < AL; ++q)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsA, (lds_void*)(base + kk * C::A_STEP + q * 4096), 16, in_k ? avo[q] : kOobOffset,
                                                 (s * KS + kk) * 128, 0, 0);
    }
    const bool in_k = s < s1 && (KS == 1 || b_col < Kb - s * C::RB);
#pragma unroll
    for (int q = 0; q < BL; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsB, (lds_void*)(base + C::A_STAGE + q * 4096), 16, in_k ? bvo[q] : kOobOffset,
                                               s * C::RB, 0, C::ONCE ? kLoadOnce : 0);
  };

  // ---- scales of a K-quad: waves 0 (and 1) 64 rows of X, 16 bytes of each, waves 2 and 3 a 64-row group of W -----------------
  using Sched = T128Schedule<NS, SPQ, C::TL>;
  static_assert(t128_covered<Sched>(), "a wait does not cover what is read behind it");
  constexpr int SD = Sched::SD, SSLOT = 4096;
  lds_u8* const sbase = smem + NS * C::STAGE;
  uint32_t sco = kOobOffset;
  if (wave < C::BM / 64) {
    if (64 * wave + lane < rows) sco = (uint32_t)(slots[64 * wave + lane] / a.replicas * a.ldxs);
  } else if (wave >= 2) {
    const int n = UP ? (wave & 1) * a.F + 64 * col : 128 * col + 64 * (wave & 1);
    if (n < a.N) sco = (uint32_t)(n / 64 * KQ * 1024 + lane * 16);
  }
  auto load_scales = [&](int Q) {
    lds_u8* const dst = sbase + Q % (SD + 1) * SSLOT + wave * 1024;
    const uint32_t vo = Q < q1 ? sco : kOobOffset;
    if (wave < 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsAs, (lds_void*)dst, 16, vo, Q * 16, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsBs, (lds_void*)dst, 16, vo, Q * 1024, 0, 0);
  };
  // X: register = row tile, byte = K-step; W: register = K-step, byte = column tile
  int sa[MT], sb[4], san[MT], sbn[4];
  const uint32_t sel = 0x0c0c0400u + (uint32_t)gq * 0x0101u;   // the lane's byte gq of each of a row's four dwords
  auto read_scales = [&](int Q) {
    lds_u8* const slot = sbase + Q % (SD + 1) * SSLOT;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const v4i x = *(lds_v4i*)(slot + (16 * MT * wm + 16 * i + r) * 16);
      const uint32_t lo = __builtin_amdgcn_perm((uint32_t)x.y, (uint32_t)x.x, sel), hi = __builtin_amdgcn_perm((uint32_t)x.w, (uint32_t)x.z, sel);
      san[i] = (int)(lo | (hi << 16));
      // two K-steps a stage, the last of them beyond K: its elements are zeros, its bytes the next row's scales (0xFF: NaN)
      if (KS == 2 && Q == KQ - 1) san[i] &= a.K % 512 ? (1 << (a.K % 512 / 16)) - 1 : -1;
    }
    if constexpr (UP) {   // tiles 0, 1: the wave's 32 rows of the gate group, 2, 3: of the up group
      const v4i g = *(lds_v4i*)(slot + 2048 + lane * 16), u = *(lds_v4i*)(slot + 3072 + lane * 16);
#pragma unroll
      for (int t = 0; t < 4; ++t)
        sbn[t] = (int)__builtin_amdgcn_perm((uint32_t)u[t], (uint32_t)g[t], wn ? 0x07060302u : 0x05040100u);
    } else {
      const v4i x = *(lds_v4i*)(slot + 2048 + wn * 1024 + lane * 16);
#pragma unroll
      for (int t = 0; t < 4; ++t) sbn[t] = x[t];
    }
  };
  auto take_scales = [&]() {
#pragma unroll
    for (int i = 0; i < MT; ++i) sa[i] = san[i];
#pragma unroll
    for (int t = 0; t < 4; ++t) sb[t] = sbn[t];
  };

  v4f acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
  v8i af[2][KS][MT], bf[2][KS][NT];
  const int swa = swz<8>(r), swb = swz<C::CPR>(r);
  auto read_a = [&](int buf, auto set, int i) {
#pragma unroll
    for (int kk = 0; kk < KS; ++kk)
      af[decltype(set)::value][kk][i] = load_frag<128, 8>(smem + buf * C::STAGE + kk * C::A_STEP + (16 * MT * wm + r) * 128, 16 * i, 0, gq, swa);
  };
  auto read_b = [&](int buf, auto set, int j) {
    lds_u8* const t = smem + buf * C::STAGE + C::A_STAGE + ((UP ? 32 : 64) * wn + bperm_lane_off(r)) * C::RB;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk)
      bf[decltype(set)::value][kk][j] = load_frag<C::RB, C::W_EB>(t, UP ? 64 * (j >> 1) + 4 * (j & 1) : bperm_tile_off(j), kk, gq, swb);
  };

  // ---- prologue ------------------------------------------------------------------------------------------------------------
#pragma unroll
  for (int k = 0; k < NS; ++k) {
    if (Sched::prologue_scales(k)) load_scales(q0 + k / SPQ);
    issue(s0 + k, k);
    __builtin_amdgcn_sched_barrier(0);               // the waits count on this order
  }
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(Sched::prologue_wait()));
  __builtin_amdgcn_sched_barrier(0);
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

  int buf = 0;                                       // buffer of stage s
  auto stage = [&](int Q, auto tc) {
    constexpr int t = decltype(tc)::value, set = t & 1;
    using Nx = std::integral_constant<int, set ^ 1>;
    const int s = Q * SPQ + t;
    if (s >= s1) return;                             // uniform
    // stage s + 1 has landed; younger are NS - 2 stages and the scales requested since
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(Sched::stage_wait(t)));
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (t == 0) {
      load_scales(Q + SD);
      __builtin_amdgcn_sched_barrier(0);
    }
    issue(s + NS, buf);
    __builtin_amdgcn_sched_barrier(0);
    const int nbuf = buf + 1 == NS ? 0 : buf + 1;
    // the next quad's scales landed before this iteration's barrier (they were requested ahead of stage s + 1)
    if constexpr (t == SPQ - 1) read_scales(Q + 1);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
      for (int j = i * NT / MT; j < (i + 1) * NT / MT; ++j) read_b(nbuf, Nx{}, j);
      read_a(nbuf, Nx{}, i);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < KS; ++kk)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = mfma_scaled<C::WF, MX_E4M3>(bf[set][kk][j], af[set][kk][i], acc[i][j], j, sb[t * KS + kk], t * KS + kk, sa[i]);
      __builtin_amdgcn_sched_barrier(0);
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

  // ---- epilogue: lane (r, gq) holds row 16 i + r, eight columns of a tile pair ------------------------------------------------
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int row = 16 * MT * wm + 16 * i + r;
    const int id = row < rows ? slots[row] : -1;
    if constexpr (UP) {
      // gate and up of columns n .. n + 7; both pass through bf16, the precision of the activation between the projections
      const int n = 64 * col + 32 * wn + 8 * gq;
      float p[8];
      uint32_t am = 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float g = bf16_to_f32(f32_to_bf16(acc[i][e / 4][e % 4])), up = bf16_to_f32(f32_to_bf16(acc[i][2 + e / 4][e % 4]));
        p[e] = silu_mul_f32(g, up);
        const uint32_t m = __builtin_bit_cast(uint32_t, p[e]) & 0x7FFFFFFFu;
        am = m > am ? m : am;
      }
#pragma unroll
      for (int d = 16; d < 64; d <<= 1) {
        const uint32_t o = (uint32_t)__shfl_xor((int)am, d);
        am = o > am ? o : am;
      }
      uint32_t code[8];
      uint8_t sbyte;
      encode_block<8>(p, am, MX_E4M3, a.scale_mode, code, sbyte);
      if (id >= 0) {
        *(uint2*)(a.q + (int64_t)id * a.F + n) = make_uint2(code[0] | (code[1] << 8) | (code[2] << 16) | (code[3] << 24),
                                                            code[4] | (code[5] << 8) | (code[6] << 16) | (code[7] << 24));
        if (gq == 0) a.qs[(int64_t)id * (a.F / 32) + n / 32] = sbyte;
      }
    } else if (id >= 0) {
      float* const c = a.C + split * a.c_split + (int64_t)id * a.N;
#pragma unroll
      for (int jp = 0; jp < 2; ++jp) {
        const int n = 128 * col + 64 * wn + 32 * jp + 8 * gq;
        store8_edge<float>(c + n, acc[i][2 * jp], acc[i][2 * jp + 1], a.N - n);
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // the trailing zero-fill DMA has left the queue before the LDS is given back
#endif
}

template <class C>
int launch(const MoeTileArgs& a, hipStream_t stream) {
  auto kern = moe_tile_kernel<C>;
  static int attr_done = 0;   // benign race: the attribute call is idempotent
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
    if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "hipFuncSetAttribute(%d bytes LDS): %s", C::LDS, hipGetErrorString(e));
    attr_done = 1;
  }
  const int64_t v = (int64_t)(C::UP ? a.F / 64 : (a.N + 127) / 128) * a.splits, blocks = (v + 7) / 8 * 8 * a.max_tiles;
  if (blocks <= 0) return MX_OK;
  if (blocks > 0x7FFFFFFF) return set_error(MX_ERR_SHAPE, "moe tile kernel: too many workgroups");
  hipError_t e = launch_kernel(kern, dim3((unsigned)blocks), dim3(256), C::LDS, stream, a);
  if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "moe_tile_kernel launch: %s", hipGetErrorString(e));
  return MX_OK;
}

}  // namespace

int launch_moe_tiles(const void* ids, int ids64, int64_t num_ids, int num_experts, int tile_rows, MoeTile* tiles, int32_t* slots, int64_t max_tiles,
                     hipStream_t stream) {
  if (num_ids < 1 || num_ids > kMoeTileMaxIds || num_experts < 1 || num_experts > kMoeTileMaxExperts)
    return set_error(MX_ERR_SHAPE, "moe tiles: unsupported sizes");
  hipError_t e = launch_kernel(moe_tiles_kernel, dim3(1), dim3(kTilesThreads), 0, stream, (const int32_t*)ids, ids64 ? 1 : 0, (int)num_ids,
                               num_experts, tile_rows, tiles, slots, (int)max_tiles);
  if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "moe_tiles_kernel launch: %s", hipGetErrorString(e));
  return MX_OK;
}

// 128 rows (only for FP4 weights, whose stages leave room for three of them) take long rows of W once where two tiles of 64 would
// read them twice.  us per layer, 64 | 128 rows: 8 experts of 4096 x 14336, 64, 80, 112 and 128 rows each 232 | 225, 263 | 229, 296 |
// 258, 332 | 318, 64 of 4096 x 1024 176 | 173, 205 | 183, 239 | 220, 269 | 262; with short rows they only pad more: 8 of 2048 x 7168
// 93 | 95 (64), 116 | 128 (128), of 1024 x 7168 64 | 70, 70 | 72, 77 | 74, 85 | 94.  FP8 (two stages of 32 KiB): 342 | 361, 370 | 370,
// 418 | 395, 456 | 453 and 79 | 85, 86 | 88, 95 | 91, 103 | 115.
int moe_tile_rows(int64_t num_ids, int64_t experts, int64_t H, int w_fmt) {
  return w_fmt == MX_E2M1 && H > 2048 && num_ids > experts * 64 ? 128 : 64;
}

// Ranges of K of the down projection: two workgroups for each of 256 CUs, from at least two K-quads each.
int moe_tile_splits(int64_t num_ids, int64_t experts, int tile_rows, int64_t N, int64_t K) {
  const int64_t used = experts < num_ids ? experts : num_ids, rows = num_ids / used;
  const int64_t wgs = used * ((rows + tile_rows - 1) / tile_rows) * ((N + 127) / 128), KQ = (K + 511) / 512;
  int64_t s = (512 + wgs / 2) / wgs;
  if (s > KQ / 2) s = KQ / 2;
  return s < 1 ? 1 : s > 8 ? 8 : (int)s;
}

int launch_moe_tile(const MoeTileArgs& a, bool up, hipStream_t stream) {
  if (a.K % 128 != 0 || (up && a.F % 64 != 0) || a.splits < 1) return set_error(MX_ERR_SHAPE, "moe tile kernel: unsupported sizes");
  // Non-temporal weights as long as nearly all experts have one tile of 64: the second one would read them from memory again.  us per layer,
  // plain | non-temporal, 40, 48, 56 and 64 rows each: 8 experts of 4096 x 14336 FP8 293 | 272, 299 | 280, 312 | 317, 342 | 399, FP4 181 |
  // 176, 187 | 182, 203 | 214, 232 | 261; 16 of 1024 x 4096 FP8 72 | 69, 73 | 70, 83 | 79, 88 | 90.
  const bool once = a.n_ids <= (int64_t)a.E * 48 &&
                    stream_loads_once((int64_t)(a.n_ids < a.E ? a.n_ids : a.E) * a.N, a.w_fmt == MX_E2M1 ? a.K / 2 : a.K, a.ldw,
                                      (uint64_t)a.W | (uint64_t)a.w_es, 1);
#define MX_CASE(WF, ROWS, ONCE, ...)                                                                                          \
  if (a.w_fmt == WF && a.tile_rows == ROWS && once == ONCE)                                                                   \
    return up ? launch<MoeTileCfg<WF, true, ROWS, ONCE, __VA_ARGS__>>(a, stream) : launch<MoeTileCfg<WF, false, ROWS, ONCE, __VA_ARGS__>>(a, stream);
  MX_CASE(MX_E4M3, 64, false, 3, 1)
  MX_CASE(MX_E4M3, 64, true, 3, 1)
  MX_CASE(MX_E2M1, 64, false, 4, 1)
  MX_CASE(MX_E2M1, 64, true, 2, 2)
  MX_CASE(MX_E2M1, 128, false, 3, 1)
#undef MX_CASE
  return set_error(MX_ERR_DTYPE, "moe tile kernel: weights must be E4M3 or E2M1");
}

}  // namespace mx
