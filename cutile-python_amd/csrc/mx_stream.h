// Interface of the weight-streaming launches (kernels in mx_gemm_stream.h).
#pragma once
#include "mx_common.h"

namespace mx {

// weight-streaming kernel (mx_gemm_stream.h): 8-bit X with plain scale rows, 8-bit or FP4 W with plain scale rows or
// scales in MX_SCALE_NATIVE, K % 128 == 0
struct StreamArgs {
  const uint8_t* X; const uint8_t* Xs; const uint8_t* W; const uint8_t* Ws; void* C;
  int32_t M, N, K;
  int64_t ldx, ldxs, ldw, ldws, ldc;   // bytes; ldc in elements; ldws unused for packed scales
  int32_t x_fmt, w_fmt, c_dtype, accumulate, ws_packed;
  // chosen by the launcher: K ranges per workgroup, row tiles, workgroups per row tile
  int32_t kw, m_tiles, units;
};
bool stream_supports(int x_fmt, int w_fmt);
// what keeps the kernel from taking a problem whose A, A_scale and unpacked B, B_scale are K-contiguous (nullptr: nothing);
// the launch refuses exactly these, so a dispatch that asks first never picks the kernel in vain
const char* stream_issue(const StreamArgs& a);
struct StreamPlan { int mt, m_tiles, nt, kw, units; float cost; };
StreamPlan stream_plan(int64_t M, int64_t N, int64_t K, int w_fmt);
int launch_gemm_stream(const StreamArgs& a, hipStream_t stream);

// mixture-of-experts layer at decode sizes (mx_moe.hip)
// Routed ids that a workgroup sorts out by itself, in a list of 4 KiB of LDS.  With room for 8192 two workgroups of the FP4
// form no longer fit on a CU and its layers take 10 - 40 % longer (8 experts of 4096 x 14336, 16 rows each: 156 -> 184 us).
// At 64 experts the limit lies about where the two forms of the layer meet (4096 x 2048, 32 rows each, streamed | grouped
// GEMMs: FP8 427 | 417 us, FP4 287 | 314); of more experts it ends the streaming early (64, 16 rows each: 318 | 403, 203 | 303).
constexpr int kMoeMaxIds = 2048;
struct MoeStreamArgs {
  const uint8_t* X; const uint8_t* Xs; const uint8_t* W; const uint8_t* Ws;
  const void* ids; const float* weights;
  uint8_t* q; uint8_t* qs; float* C;   // up: elements and scales [n_ids][F]; down: [n_ids][N]
  int64_t ldx, ldxs, ldw, ldws, w_es, ws_es;   // bytes; *_es: between experts
  int32_t x_rows, N, K, F;             // N: rows of an expert's W (up: 2 F)
  int32_t n_ids, ids64, E, replicas;   // a routed copy `id` reads row id / replicas of X
  int32_t w_fmt, ws_packed, scale_mode;
  int32_t kw, units;                   // chosen by the launcher
};
int launch_moe_stream(const MoeStreamArgs& a, bool up, hipStream_t stream);
int launch_moe_combine(const float* c, int splits, int64_t c_split, const float* weights, const void* ids, int ids64, int E, int64_t T, int topk, int64_t H, void* out,
                       int out_dtype, hipStream_t stream);

}  // namespace mx
