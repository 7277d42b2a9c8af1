// Launches of the weight-streaming kernel (mx_gemm_stream.h) for plain products.
#include "mx_gemm_stream.h"

namespace mx {
namespace {

// Workgroup of C::WAVES waves: kw K ranges x WAVES / kw units of NT tiles.  m_tiles row tiles of 16 MT rows are neighbours in
// dispatch order on the same XCD (workgroup ids go round-robin over 8 XCDs), so W is read from memory once.
template <class C>
__global__ __launch_bounds__(C::WAVES * 64) void stream_kernel(const StreamArgs a) {
  constexpr int NT = C::NT, MT = C::MT;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem_generic[];
  lds_u8* const smem = (lds_u8*)smem_generic;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, gq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kq = wave % a.kw, nw = wave / a.kw, nwv = C::WAVES / a.kw;
  int unit0 = blockIdx.x, mt = 0;
  if (a.m_tiles > 1) {
    const int per = 8 * a.m_tiles, hi = unit0 / per, in = unit0 % per;
    mt = in / 8;
    unit0 = hi * 8 + in % 8;
    if (unit0 >= a.units) return;   // uniform: the grid is rounded up to whole rows of 8
  }
  const int m0 = mt * 16 * MT;
  const int u = unit0 * nwv + nw;                    // unit of NT tiles
  const int G = u * NT / 4, j0[1] = {u * NT % 4};
  const int KQ = (a.K + 511) / 512;
  const int Q0 = kq * KQ / a.kw, Q1 = (kq + 1) * KQ / a.kw;

  StreamWave w;
  w.rsX = make_rsrc(a.X, (uint32_t)((int64_t)(a.M - 1) * a.ldx + a.K));
  w.rsXs = make_rsrc(a.Xs, (uint32_t)((int64_t)(a.M - 1) * a.ldxs + a.K / 32));
  w.rsW = make_rsrc(a.W, (uint32_t)((int64_t)(a.N - 1) * a.ldw + (int64_t)a.K * (C::WF == MX_E2M1 ? 1 : 2) / 2));
  w.rsWs = C::PACKED ? make_rsrc(a.Ws, (uint32_t)(packed_scale_dwords(a.N, a.K) * 4))
                     : make_rsrc(a.Ws, (uint32_t)((int64_t)(a.N - 1) * a.ldws + a.K / 32));
  uint32_t xvo[2 * MT], xso[MT], wvo[2 * NT], wso[C::NSW];
#pragma unroll
  for (int q = 0; q < 2 * MT; ++q) {
    const int m = m0 + 8 * q + (lane >> 3);
    xvo[q] = m < a.M ? (uint32_t)(m * a.ldx + stream_x_col(q, lane)) : kOobOffset;
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = m0 + 16 * i + r;
    xso[i] = m < a.M ? (uint32_t)(m * a.ldxs) : kOobOffset;
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = 64 * G + bperm_row(j0[0] + j, r);
    if constexpr (!C::PACKED) wso[j] = n < a.N ? (uint32_t)(n * a.ldws) : kOobOffset;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int nl = 64 * G + bperm_row(j0[0] + j, 8 * h + (lane >> 3));
      wvo[2 * j + h] = nl < a.N ? (uint32_t)(nl * a.ldw + (lane & 7) * 16) : kOobOffset;
    }
  }
  if constexpr (C::PACKED) wso[0] = 64 * G < a.N ? (uint32_t)(G * KQ * 1024 + lane * 16) : kOobOffset;

  v4f acc[MT][NT];
  stream_products<C>(w, smem + wave * C::WAVE_BYTES, xvo, xso, wvo, wso, j0, Q0, Q1, (a.K + 127) / 128, acc);

  // ---- the K ranges meet in LDS, added in their order ------------------------------------------------------------
  __syncthreads();
  typedef __attribute__((address_space(3))) v4f lds_v4f;
  lds_v4f* const red = (lds_v4f*)smem;               // [nw][kq][i][j][lane]
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) red[((nw * a.kw + kq) * (MT * NT) + i * NT + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  // item = (unit, row tile, tile pair) of the workgroup; lane (c, g) of tile j holds row c, columns
  // bperm_tile_off(j) + 8 g .. + 3 of the group, so a pair of tiles is 8 consecutive outputs of a lane
  constexpr int JP = NT >= 2 ? 2 : 1;
  for (int it = wave; it < nwv * MT * (NT / JP); it += C::WAVES) {   // uniform per wave
    const int jp = it % (NT / JP), i = it / (NT / JP) % MT, wv = it / (NT / JP) / MT;
    v4f v[2] = {};
    for (int k = 0; k < a.kw; ++k)
#pragma unroll
      for (int h = 0; h < JP; ++h) v[h] += red[((wv * a.kw + k) * (MT * NT) + i * NT + jp * JP + h) * 64 + lane];
    const int t0 = (unit0 * nwv + wv) * NT + jp * JP;                     // first tile of the item
    const int n = 64 * (t0 / 4) + bperm_tile_off(t0 % 4) + 8 * gq, m = m0 + 16 * i + r;
    int cols = a.N - n;
    if (JP == 1 && cols > 4) cols = 4;
    if (m < a.M && cols > 0) {
      if (a.c_dtype == MX_F32) {
        float* p = (float*)a.C + (int64_t)m * a.ldc + n;
        if (a.accumulate) add8_edge<float>(p, v[0], v[1], cols);
        store8_edge<float>(p, v[0], v[1], cols);
      } else {
        uint16_t* p = (uint16_t*)a.C + (int64_t)m * a.ldc + n;
        if (a.accumulate) add8_edge<uint16_t>(p, v[0], v[1], cols);
        store8_edge<uint16_t>(p, v[0], v[1], cols);
      }
    }
  }
}

// Waves of a workgroup: with 64 rows of X a stage of FP4 weights is 16 KiB of X, of which two for each of 8 waves do not fit
// into LDS.
constexpr int stream_waves(int mt, int w_fmt) { return mt == 4 && w_fmt == MX_E2M1 ? 4 : 8; }

template <class C>
int launch(const StreamArgs& a, int blocks, hipStream_t stream) {
  auto kern = stream_kernel<C>;
  static int attr_done = 0;   // benign race: the attribute call is idempotent
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES);
    if (e != hipSuccess)
      return set_error(MX_ERR_LAUNCH, "hipFuncSetAttribute(%d bytes LDS): %s", C::LDS_BYTES, hipGetErrorString(e));
    attr_done = 1;
  }
  hipError_t e = launch_kernel(kern, dim3((unsigned)blocks), dim3(C::WAVES * 64), C::LDS_BYTES, stream, a);
  if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "stream_kernel launch: %s", hipGetErrorString(e));
  return MX_OK;
}

template <int XF, int WF, int NT, int MT>
int launch_p(const StreamArgs& a, int blocks, hipStream_t stream) {
  constexpr int W = stream_waves(MT, WF);
  if constexpr (NT == 4)
    if (stream_loads_once(a.N, WF == MX_E2M1 ? a.K / 2 : a.K, a.ldw, (uint64_t)a.W, a.m_tiles))
      return a.ws_packed ? launch<StreamCfg<XF, WF, NT, MT, true, W, false, true>>(a, blocks, stream)
                         : launch<StreamCfg<XF, WF, NT, MT, false, W, false, true>>(a, blocks, stream);
  return a.ws_packed ? launch<StreamCfg<XF, WF, NT, MT, true, W>>(a, blocks, stream)
                     : launch<StreamCfg<XF, WF, NT, MT, false, W>>(a, blocks, stream);
}
template <int XF, int WF, int NT>
int launch_m(const StreamArgs& a, int mt, int blocks, hipStream_t stream) {
  return mt == 1 ? launch_p<XF, WF, NT, 1>(a, blocks, stream)
         : mt == 2 ? launch_p<XF, WF, NT, 2>(a, blocks, stream) : launch_p<XF, WF, NT, 4>(a, blocks, stream);
}

}  // namespace

bool stream_supports(int x_fmt, int w_fmt) {
  return (x_fmt == MX_E4M3 && (w_fmt == MX_E4M3 || w_fmt == MX_E2M1)) ||
         (x_fmt == MX_E5M2 && (w_fmt == MX_E5M2 || w_fmt == MX_E2M1));
}

// How the waves of a workgroup split the problem: kw K ranges x waves / kw units of nt tiles; M in tiles of 16 mt rows.  The
// cost that is minimised is a wave's K-quads times what a K-step of it moves (nt tiles of W, the rows of X), plus a
// start-up per workgroup, for every round of workgroups over the 256 CUs: X is fetched once per unit, so wide units
// save traffic, but a second, partly filled round costs more (28672 x 8192 FP4 at 4 rows: 224 workgroups 28 us, 448
// 33.6 us; 14336 x 8192 FP8 at 64 rows: 224 of 4 tiles 34 us, 448 of 2 45 us).
// (tiles of a 64-row group interleave its rows, so groups are covered whole)
StreamPlan stream_plan(int64_t M, int64_t N, int64_t K, int w_fmt) {
  StreamPlan p = {};
  // FP4 weights for 33 .. 64 rows: one row tile of 64 (four waves) once the weights have 8192 rows to share out, which
  // reads them once (28672 x 8192: 64 rows 52.6 -> 44.8 us, 48 rows 47.9 -> 41.7; 14336 x 4096, 40 rows 16.1 -> 15.0);
  // with fewer, two tiles of 32 have the waves that it lacks (4096 x 14336, 64 rows: 17.8 against 21.5)
  p.mt = M <= 16 ? 1 : M <= 32 ? 2 : w_fmt != MX_E2M1 ? 4 : M <= 64 && N >= 8192 ? 4 : 2;
  const int waves = stream_waves(p.mt, w_fmt);   // (half as many waves have twice the bandwidth each)
  p.m_tiles = (int)((M + 16 * p.mt - 1) / (16 * p.mt));
  const int tiles = (int)((N + 63) / 64 * 4), KQ = (int)((K + 511) / 512);
  const float wb = w_fmt == MX_E2M1 ? 1.f : 2.f, xb = (M < 16 * p.mt ? M : 16 * p.mt) / 16.f;
  p.cost = 1e30f;
  for (int n = 4; n >= 1; n >>= 1)
    for (int kw = waves; kw >= 1; kw >>= 1) {
      if (kw > 1 && kw > KQ) continue;
      const int units = (tiles + n * (waves / kw) - 1) / (n * (waves / kw));
      const int64_t rounds = ((int64_t)units * p.m_tiles + 255) / 256;
      const float t = rounds * ((KQ + kw - 1) / kw * (n * wb + xb) * waves / 8.f + 3.f);
      if (t < p.cost) { p.cost = t; p.nt = n; p.kw = kw; p.units = units; }
    }
  return p;
}

// Rows may overlap (a row pitch of zero is a broadcast row): the descriptors end behind the last row's last byte.
const char* stream_issue(const StreamArgs& a) {
  if (!stream_supports(a.x_fmt, a.w_fmt)) return "it takes 8-bit A with FP4 B or B of A's format";
  if (a.K < 128 || a.K % 128 != 0) return "K is not a multiple of 128";
  if ((((uintptr_t)a.X | (uintptr_t)a.W | (uintptr_t)a.ldx | (uintptr_t)a.ldw) % 16) != 0)
    return "A and B must have 16-byte aligned rows";
  if ((((uintptr_t)a.Xs | (uintptr_t)a.ldxs) % 4) != 0) return "A_scale must have 4-byte aligned rows";
  if (a.ws_packed ? ((uintptr_t)a.Ws % 16) != 0 : (((uintptr_t)a.Ws | (uintptr_t)a.ldws) % 4) != 0)
    return "B_scale must be 16-byte aligned (packed) or have 4-byte aligned rows";
  // lane offsets are 32-bit, and 2^31 marks what does not exist
  auto fits = [](int64_t rows, int64_t pitch, int64_t row) {
    return rows * pitch < (int64_t)1 << 31 && (rows - 1) * pitch + row < (int64_t)1 << 31;
  };
  if (!fits(a.M, a.ldx, a.K) || !fits(a.N, a.ldw, a.w_fmt == MX_E2M1 ? a.K / 2 : a.K)) return "A or B spans 2 GiB or more";
  if (!fits(a.M, a.ldxs, a.K / 32) ||
      !(a.ws_packed ? fits(1, 0, packed_scale_dwords(a.N, a.K) * 4) : fits(a.N, a.ldws, a.K / 32)))
    return "A_scale or B_scale spans 2 GiB or more";
  return nullptr;
}

int launch_gemm_stream(const StreamArgs& a0, hipStream_t stream) {
  StreamArgs a = a0;
  if (a.M < 1 || a.N < 1) return set_error(MX_ERR_SHAPE, "stream kernel: no rows");
  if (const char* why = stream_issue(a)) return set_error(MX_ERR_LAYOUT, "stream kernel: %s", why);
  const StreamPlan p = stream_plan(a.M, a.N, a.K, a.w_fmt);
  const int mt = p.mt, nt = p.nt;
  a.m_tiles = p.m_tiles; a.kw = p.kw; a.units = p.units;
  const int blocks = a.m_tiles > 1 ? (a.units + 7) / 8 * 8 * a.m_tiles : a.units;
#define MX_CASE(XF, WF)                                                                       \
  if (a.x_fmt == XF && a.w_fmt == WF)                                                         \
    return nt == 4 ? launch_m<XF, WF, 4>(a, mt, blocks, stream)                               \
           : nt == 2 ? launch_m<XF, WF, 2>(a, mt, blocks, stream) : launch_m<XF, WF, 1>(a, mt, blocks, stream);
  MX_CASE(MX_E4M3, MX_E4M3)
  MX_CASE(MX_E4M3, MX_E2M1)
  MX_CASE(MX_E5M2, MX_E5M2)
  MX_CASE(MX_E5M2, MX_E2M1)
#undef MX_CASE
  return MX_ERR_DTYPE;
}

}  // namespace mx
