// Interface of the 128 x 128 one-tile kernel (mx_gemm_t128.hip): small and mid-size products, batches of them, lists of
// unequal ones, split-K, and the grouped form with 128-slot tiles.
#pragma once
#include "mx_common.h"

namespace mx {

constexpr int kT128ScalesAny = 2;   // a_plain, b_plain: rows at any byte

struct T128Args {
  const uint8_t* A;        // [M rows][lda bytes], K contiguous
  const uint8_t* B;        // [N rows][ldb bytes]
  const uint8_t* As;       // a_plain: [M rows][ldas bytes]; else the native layout (operand A, slot order when grouped)
  const uint8_t* Bs;       // b_plain: [N rows][ldbs bytes]; else the native layout (operand B)
  void* C;
  const float* acc;        // what is added to the product (fp32, laid out like C); null: C itself if `accumulate`
  int64_t lda, ldb, ldas, ldbs, ldc;   // bytes; ldc in elements
  int64_t a_batch, b_batch, as_batch, bs_batch, c_batch;   // from one product of a batch to the next: bytes, elements of C
  float* partial;          // k_splits > 1: fp32 partial products [split][M][N]
  int32_t M, N, K;
  int32_t a_fmt, b_fmt, c_dtype, accumulate;
  int32_t a_plain, b_plain;            // 0, 1, or kT128ScalesAny (both)
  int32_t batch, k_splits; // 1 each unless used
  // grouped (MoE) extension; sorted_token_ids == nullptr otherwise.  M is the number of slots.
  const int32_t* sorted_token_ids;
  const int32_t* sorted_expert_ids;
  const float* topk_weights;
  int32_t tile_m, replicas, num_experts;
  int64_t num_valid_ids, a_rows, b_expert, bs_expert;      // rows of A; bytes between experts
};

// scales that the kernel reads where they are: K-contiguous rows of 4-byte aligned E8M0 bytes, K a whole number of stages
inline bool t128_plain_scales(const void* ptr, int64_t ld, int64_t k_stride, int64_t rows, int64_t K, int a_fmt, int b_fmt) {
  const int stage = a_fmt == MX_E2M1 && b_fmt == MX_E2M1 ? 256 : 128;
  return k_stride == 1 && K % stage == 0 && ld % 4 == 0 && ((uintptr_t)ptr) % 4 == 0 && rows * ld < ((int64_t)1 << 31) &&
         (rows - 1) * ld + K / 32 < ((int64_t)1 << 31);
}
// ... and rows that it fetches dword by dword (kT128ScalesAny): K-contiguous, whatever their alignment and wherever K ends
inline bool t128_any_scales(int64_t ld, int64_t k_stride, int64_t rows, int64_t K) {
  const int64_t lim = ((int64_t)1 << 31) - 64;   // (the last quad's window reaches beyond its row)
  return k_stride == 1 && K >= 32 && rows * ld < lim && (rows - 1) * ld + K / 32 < lim;
}
// ... where that is the faster way: it costs every stage of every tile, the re-layout launch costs a call 3 .. 4 us.  MXFP8 (any | re-
// laid first): 1024 x 1024 x 5440 18.9 | 21.6 us, 2048 x 2048 x 5440 35.1 | 36.0, 3072 x 1500 x 4000 (9216 stages) 41.6 | 41.3, x 5440
// 51.7 | 47.0, 5653 x 944 x 5440 49.2 | 46.9; MXFP4: 2048 x 2048 x 5440 25.7 | 26.4, 3072 x 1500 x 4000 (4608) 28.7 | 29.4, x 5440
// 35.0 | 33.7.
inline bool t128_any_pays(int64_t M, int64_t N, int64_t K, int64_t batch, bool fp4) {
  const int64_t stages = (K + (fp4 ? 255 : 127)) / (fp4 ? 256 : 128);
  return ((M + 127) / 128) * ((N + 127) / 128) * batch * stages <= (fp4 ? 4800 : 10000);
}
// 64 x 64 tiles of a product; up to kT128SmallTiles workgroups (two for every CU) of them run instead of 128 x 128 ones
// (measured either side in mx_gemm_t128.hip)
constexpr int64_t kT128SmallTiles = 512;
inline int64_t t128_small_tiles(int64_t M, int64_t N) { return ((M + 63) / 64) * ((N + 63) / 64); }
int launch_gemm_t128(const T128Args& g, hipStream_t stream);
// any number of independent plain products of one element-format pair: one persistent launch per 32 of them
int launch_gemm_t128_list(const T128Args* problems, int n, hipStream_t stream);

}  // namespace mx
