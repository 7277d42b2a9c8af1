// Mixture-of-experts layer at decode sizes (a few rows per expert) and the pass that adds the top-k copies.
//
// Bound: reading the touched experts' weights once.  At these sizes a grouped GEMM on 256 x 256 tiles spends its time
// on rows that are not there, and the passes around it (alignment of the routed ids, bf16 activation out and in,
// quantisation, clearing and converting the copies) are launches of a few us each.  Here the layer is three launches:
//   moe_stream_kernel<UP>:   gate and up projection of one 32-column block per wave (mx_gemm_stream.h), SiLU(gate) * up and
//                            the MX quantisation of the product in the epilogue, where the block's 32 columns lie in
//                            the four lanes of a row;
//   moe_stream_kernel<DOWN>: down projection times the routed weight, fp32, one row per routed copy;
//   moe_combine_kernel:      the sum of a token's copies.
// Every workgroup finds the rows of its expert itself: it reads the routed ids (at most 2048: 8 KiB or 16 KiB out of L2)
// while nothing else could run in its place, so no alignment launch and no slot arrays are needed.
#include "mx_gemm_stream.h"
#include "mx_quant.h"

namespace mx {
namespace {

template <class C>
__global__ __launch_bounds__(C::WAVES * 64, 2) void moe_stream_kernel(const MoeStreamArgs a) {
  constexpr int NT = C::NT, MT = C::MT, ROWS = 16 * MT, NTHR = C::WAVES * 64;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem_generic[];
  lds_u8* const smem = (lds_u8*)smem_generic;
  typedef __attribute__((address_space(3))) uint16_t lds_u16;
  typedef __attribute__((address_space(3))) int lds_int;
  lds_u16* const list = (lds_u16*)(smem + C::LDS_BYTES);              // the expert's routed copies, in order
  lds_int* const wcnt = (lds_int*)(smem + C::LDS_BYTES + kMoeMaxIds * 2);   // per wave: ids found
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, gq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int expert = blockIdx.x / a.units, unit0 = blockIdx.x % a.units;

  // ---- rows of this expert: ids in rounds of one per thread, kept in their order -------------------------------
  int cnt = 0;
  for (int i0 = 0; i0 < a.n_ids; i0 += NTHR) {
    const int i = i0 + tid;
    int e = -1;
    if (i < a.n_ids) e = a.ids64 ? (int)((const int64_t*)a.ids)[i] : ((const int32_t*)a.ids)[i];
    const uint64_t m = __builtin_amdgcn_ballot_w64(e == expert);
    if (lane == 0) wcnt[wave] = __builtin_popcountll(m);
    __syncthreads();
    int base = cnt;
    for (int w = 0; w < C::WAVES; ++w) {
      const int c = wcnt[w];
      if (w < wave) base += c;
      cnt += c;
    }
    if (e == expert) list[base + __builtin_popcountll(m & ((1ull << lane) - 1))] = (uint16_t)i;
    __syncthreads();
  }
  cnt = __builtin_amdgcn_readfirstlane(cnt);
  if (cnt == 0) return;                              // uniform per workgroup

  const int kq = wave % a.kw, nw = wave / a.kw, nwv = C::WAVES / a.kw;
  const int u = unit0 * nwv + nw;
  const int KQ = (a.K + 511) / 512;
  const int Q0 = kq * KQ / a.kw, Q1 = (kq + 1) * KQ / a.kw;
  // first row of tiles 0, 1 and of tiles 2, 3 of the wave (32 rows each)
  const int half[2] = {C::UP ? 32 * u : 64 * u, C::UP ? a.F + 32 * u : 64 * u + 32};
  const int n_end = C::UP ? a.F : a.N;               // columns of a half that exist

  StreamWave w;
  w.rsX = make_rsrc(a.X, (uint32_t)((int64_t)(a.x_rows - 1) * a.ldx + a.K));
  w.rsXs = make_rsrc(a.Xs, (uint32_t)((int64_t)(a.x_rows - 1) * a.ldxs + a.K / 32));
  w.rsW = make_rsrc(a.W + (int64_t)expert * a.w_es, (uint32_t)((int64_t)(a.N - 1) * a.ldw + (int64_t)a.K * (C::WF == MX_E2M1 ? 1 : 2) / 2));
  w.rsWs = make_rsrc(a.Ws + (int64_t)expert * a.ws_es, C::PACKED ? (uint32_t)(packed_scale_dwords(a.N, a.K) * 4)
                                                                 : (uint32_t)((int64_t)(a.N - 1) * a.ldws + a.K / 32));
  uint32_t wvo[2 * NT], wso[C::NSW];
  int j0[C::UP ? 2 : 1];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int base = half[j / 2] + 4 * (j % 2);
    const bool in = (C::UP ? 32 * u : half[j / 2]) < n_end;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int nl = base + bperm_lane_off(8 * h + (lane >> 3));
      wvo[2 * j + h] = in && nl < a.N ? (uint32_t)(nl * a.ldw + (lane & 7) * 16) : kOobOffset;
    }
    if constexpr (!C::PACKED) {
      const int n = base + bperm_lane_off(r);
      wso[j] = in && n < a.N ? (uint32_t)(n * a.ldws) : kOobOffset;
    }
  }
#pragma unroll
  for (int g = 0; g < (C::UP ? 2 : 1); ++g) {
    j0[g] = half[g] / 32 % 2 * 2;
    if constexpr (C::PACKED) wso[g] = half[g] < a.N ? (uint32_t)(half[g] / 64 * KQ * 1024 + lane * 16) : kOobOffset;
  }

  for (int c0 = 0; c0 < cnt; c0 += ROWS) {           // uniform per workgroup; one pass unless the routing is skewed
    uint32_t xvo[2 * MT], xso[MT];
#pragma unroll
    for (int q = 0; q < 2 * MT; ++q) {
      const int s = c0 + 8 * q + (lane >> 3);
      xvo[q] = s < cnt ? (uint32_t)(list[s] / a.replicas * a.ldx + stream_x_col(q, lane)) : kOobOffset;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int s = c0 + 16 * i + r;
      xso[i] = s < cnt ? (uint32_t)(list[s] / a.replicas * a.ldxs) : kOobOffset;
    }
    v4f acc[MT][NT];
    stream_products<C>(w, smem + wave * C::WAVE_BYTES, xvo, xso, wvo, wso, j0, Q0, Q1, (a.K + 127) / 128, acc);

    // ---- the K ranges meet in LDS, added in their order ----------------------------------------------------------
    __syncthreads();
    typedef __attribute__((address_space(3))) v4f lds_v4f;
    lds_v4f* const red = (lds_v4f*)smem;             // [nw][kq][i][j][lane]
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) red[((nw * a.kw + kq) * (MT * NT) + i * NT + j) * 64 + lane] = acc[i][j];
    __syncthreads();
    for (int it = wave; it < nwv * MT * (C::UP ? 1 : 2); it += C::WAVES) {   // uniform per wave
      const int jp = C::UP ? 0 : it % 2, rest = C::UP ? it : it / 2, i = rest % MT, wv = rest / MT;
      constexpr int JN = C::UP ? 4 : 2;
      v4f v[JN] = {};
      for (int k = 0; k < a.kw; ++k)
#pragma unroll
        for (int h = 0; h < JN; ++h) v[h] += red[((wv * a.kw + k) * (MT * NT) + i * NT + jp * 2 + h) * 64 + lane];
      const int s = c0 + 16 * i + r, id = s < cnt ? (int)list[s] : -1;
      const int un = unit0 * nwv + wv;
      if constexpr (C::UP) {
        // lane (row, gq): gate and up of columns 32 un + 8 gq .. + 7; both pass through bf16, the precision of the
        // activation between the projections
        const int n = 32 * un + 8 * gq;
        float p[8];
        uint32_t am = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float g = bf16_to_f32(f32_to_bf16(v[e / 4][e % 4])), up = bf16_to_f32(f32_to_bf16(v[2 + e / 4][e % 4]));
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
        uint8_t sb;
        encode_block<8>(p, am, MX_E4M3, a.scale_mode, code, sb);
        if (id >= 0 && n < a.F) {
          *(uint2*)(a.q + (int64_t)id * a.F + n) =
              make_uint2(code[0] | (code[1] << 8) | (code[2] << 16) | (code[3] << 24),
                         code[4] | (code[5] << 8) | (code[6] << 16) | (code[7] << 24));
          if (gq == 0) a.qs[(int64_t)id * (a.F / 32) + un] = sb;
        }
      } else {
        const int n = 64 * un + 32 * jp + 8 * gq, cols = a.N - n;
        if (id >= 0 && cols > 0) {
          const float wt = a.weights ? a.weights[id] : 1.f;
          store8_edge<float>(a.C + (int64_t)id * a.N + n, v[0] * wt, v[1] * wt, cols);
        }
      }
    }
    __syncthreads();                                 // the sums are read before the next rows' stages overwrite them
  }
}

// out[t, :] = sum over the top-k copies of a token, in their order; a copy whose expert id is outside [0, E) was never
// computed and counts as zero.  A copy is the sum of `splits` partial products, c_split elements apart, times its routed weight
// (null: c holds the weighted ones).  Four columns per thread, whole waves per token, KU copies requested at a time.
// Bound: reading the copies.  Against a thread for every four columns of all tokens, which takes a 64-bit division each and waits for one
// copy after the other: 4096 tokens x 2 copies of 4096 behind the MoE layer's product 33.6 -> 31.2 us (6.4 TB/s), 3500 x 4 of 2048 22.3 ->
// 20.4, 8192 x 4 of 2048 53.4 -> 44.2, 300 x 8 of 2048 7.0 -> 5.6; columns that leave part of a wave idle cost what is idle: 6000 x 2 of 1028 11.7 ->
// 13.2, of 2560 columns 31.0 -> 32.6.  (Four copies at a time: 23.5 for the second.  Workgroups of five waves 34.6 for the last, whole threads
// counted over all columns with a 32-bit division 35.3; rows that are not whole 16-byte pieces, two copies at a time: 3000 x 3 of 1030 14.2 | 16.7.)
template <int KU>
__global__ __launch_bounds__(256) void moe_combine_kernel(const float* __restrict__ c, int splits, int64_t c_split,
                                                          const float* __restrict__ weights, const void* __restrict__ ids, int ids64,
                                                          int E, int64_t T, int topk, int64_t H, void* out, int out_dtype) {
  // (the parts of a token next to each other: they share lines where its rows don't start at one)
  const int64_t t = ((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * blockDim.y + __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int64_t h = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (t >= T || h >= H) return;
  const int n = H - h < 4 ? (int)(H - h) : 4;
  const bool whole = n == 4 && (H & 3) == 0;
  v4f s = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < topk; k0 += KU) {
    v4f v[KU];
#pragma unroll
    for (int j = 0; j < KU; ++j) v[j] = (v4f){0.f, 0.f, 0.f, 0.f};
    for (int sp = 0; sp < splits; ++sp) {
      v4f x[KU];
#pragma unroll
      for (int j = 0; j < KU; ++j) {
        // (a dropped copy's memory is read as well, and left out below)
        const float* p = c + sp * c_split + (t * topk + (k0 + j < topk ? k0 + j : topk - 1)) * H + h;
        x[j] = (v4f){0.f, 0.f, 0.f, 0.f};
        if (whole) x[j] = *(const v4f*)p;
        else
          for (int e = 0; e < n; ++e) x[j][e] = p[e];
      }
#pragma unroll
      for (int j = 0; j < KU; ++j) v[j] += x[j];
    }
#pragma unroll
    for (int j = 0; j < KU; ++j) {
      if (k0 + j >= topk) break;                     // uniform, as the next one
      const int64_t id = t * topk + k0 + j;
      const int e = ids64 ? (int)((const int64_t*)ids)[id] : ((const int32_t*)ids)[id];
      if (e < 0 || e >= E) continue;
      s += weights ? v[j] * weights[id] : v[j];
    }
  }
  if (out_dtype == MX_F32) store8_edge<float>((float*)out + t * H + h, s, s, n);
  else store8_edge<uint16_t>((uint16_t*)out + t * H + h, s, s, n);
}

template <class C>
int launch(const MoeStreamArgs& a, int blocks, hipStream_t stream) {
  auto kern = moe_stream_kernel<C>;
  constexpr int lds = C::LDS_BYTES + kMoeMaxIds * 2 + 64;
  static int attr_done = 0;   // benign race: the attribute call is idempotent
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "hipFuncSetAttribute(%d bytes LDS): %s", lds, hipGetErrorString(e));
    attr_done = 1;
  }
  hipError_t e = launch_kernel(kern, dim3((unsigned)blocks), dim3(C::WAVES * 64), lds, stream, a);
  if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "moe_stream_kernel launch: %s", hipGetErrorString(e));
  return MX_OK;
}

template <int WF, bool PACKED, bool UP>
int launch_mt(const MoeStreamArgs& a, int mt, int blocks, hipStream_t stream) {
  // Non-temporal weights up to 24 rows per expert (experts that no id names are not read): beyond, experts get more rows than a
  // pass takes and read W again.  us per layer, plain | non-temporal, rows per expert 22, 24, 28, 32: 16 experts of 4096 x 4096
  // FP8 161 | 142, 179 | 171, 192 | 191, 216 | 227; 8 of 4096 x 14336 FP4 157 | 149, 182 | 180, 184 | 183, 214 | 227, FP8 257 |
  // 234, 284 | 276, 293 | 278, 353 | 348; 32 of 2048 x 2048 FP8 24, 28, 32 rows 103.6 | 99, 117.4 | 119.3, 126 | 135; 64 of them FP4
  // 140 | 138, 146 | 149, 166 | 173.
  const int64_t rows = (int64_t)(a.n_ids < a.E ? a.n_ids : a.E) * a.N;
  if (a.n_ids <= (int64_t)a.E * 24 && stream_loads_once(rows, WF == MX_E2M1 ? a.K / 2 : a.K, a.ldw, (uint64_t)a.W | (uint64_t)a.w_es, 1))
    return mt == 1 ? launch<StreamCfg<MX_E4M3, WF, 4, 1, PACKED, 4, UP, true>>(a, blocks, stream)
                   : launch<StreamCfg<MX_E4M3, WF, 4, 2, PACKED, 4, UP, true>>(a, blocks, stream);
  return mt == 1 ? launch<StreamCfg<MX_E4M3, WF, 4, 1, PACKED, 4, UP>>(a, blocks, stream)
                 : launch<StreamCfg<MX_E4M3, WF, 4, 2, PACKED, 4, UP>>(a, blocks, stream);
}

}  // namespace

int launch_moe_stream(const MoeStreamArgs& a0, bool up, hipStream_t stream) {
  MoeStreamArgs a = a0;
  if (a.w_fmt != MX_E4M3 && a.w_fmt != MX_E2M1) return set_error(MX_ERR_DTYPE, "moe stream kernel: weights must be E4M3 or E2M1");
  if (a.n_ids < 1 || a.n_ids > kMoeMaxIds || a.K % 128 != 0 || (up && a.F % 32 != 0))
    return set_error(MX_ERR_SHAPE, "moe stream kernel: unsupported sizes");
  constexpr int waves = 4;
  const int KQ = (a.K + 511) / 512;
  // two K ranges keep every wave a few K-quads long (a workgroup's start and its tail are not hidden by its own
  // waves), four where K is long
  a.kw = KQ >= 16 ? 4 : KQ >= 2 ? 2 : 1;
  const int nwv = waves / a.kw, cols = up ? a.F / 32 : (a.N + 63) / 64;
  a.units = (cols + nwv - 1) / nwv;
  const int64_t blocks = (int64_t)a.units * a.E;
  if (blocks > 0x7FFFFFFF) return set_error(MX_ERR_SHAPE, "moe stream kernel: too many workgroups");
  // rows per pass: 16 as long as an expert is expected to get fewer than that, else 32
  const int mt = (int64_t)a.n_ids * 2 <= (int64_t)a.E * 16 ? 1 : 2;
#define MX_CASE(WF)                                                                                              \
  if (a.w_fmt == WF)                                                                                             \
    return a.ws_packed ? (up ? launch_mt<WF, true, true>(a, mt, (int)blocks, stream)                              \
                             : launch_mt<WF, true, false>(a, mt, (int)blocks, stream))                            \
                       : (up ? launch_mt<WF, false, true>(a, mt, (int)blocks, stream)                             \
                             : launch_mt<WF, false, false>(a, mt, (int)blocks, stream));
  MX_CASE(MX_E4M3)
  MX_CASE(MX_E2M1)
#undef MX_CASE
  return MX_ERR_DTYPE;
}

int launch_moe_combine(const float* c, int splits, int64_t c_split, const float* weights, const void* ids, int ids64, int E, int64_t T, int topk, int64_t H, void* out,
                       int out_dtype, hipStream_t stream) {
  if (T <= 0 || H <= 0) return MX_OK;
  // A token's columns in parts of one, two or four waves, as few idle lanes as can be and then as long as can be; workgroups of four waves, several
  // tokens together, where that leaves two for each CU.
  const int64_t h4 = (H + 3) / 4;
  int64_t threads = 256;
  for (int64_t n = 128; n >= 64; n /= 2)
    if ((h4 + n - 1) / n * n < (h4 + threads - 1) / threads * threads) threads = n;
  const int64_t parts = (h4 + threads - 1) / threads, tokens = T * parts >= 512 * (256 / threads) ? 256 / threads : 1;
  const int64_t groups = (T + tokens - 1) / tokens, z = (groups + 65534) / 65535;   // (a grid has less than 65536 of y and z)
  const dim3 grid((unsigned)parts, (unsigned)((groups + z - 1) / z), (unsigned)z), block((unsigned)threads, (unsigned)tokens);
  auto run = [&](auto kern) { return launch_kernel(kern, grid, block, 0, stream, c, splits, c_split, weights, ids, ids64, E, T, topk, H, out,
                                                             out_dtype); };
  hipError_t e = topk == 1 || H % 4 != 0 ? run(moe_combine_kernel<1>) : run(moe_combine_kernel<2>);
  if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "moe_combine_kernel launch: %s", hipGetErrorString(e));
  return MX_OK;
}

}  // namespace mx
