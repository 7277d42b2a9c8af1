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
int launch_gemm_stream(const StreamArgs& a, hipStream_t stream);

}  // namespace mx
