// C ABI of libmxgemm.so: argument validation and kernel dispatch.  See include/mxgemm.h.
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <vector>

#include "mx_common.h"
#include "mx_gemm_pp.h"
#include "mx_gemm_t128.h"
#include "mx_moe_rules.h"
#include "mx_moe_tile.h"
#include "mx_stream.h"

// Scratch of mx_gemm_static: lives in the library's device image, one copy per GPU the library runs on, held
// until the process ends.  Host code never uses this name as an address: static_scratch() below resolves the
// device address once per device with hipGetSymbolAddress and everything else uses that pointer.
static __device__ __align__(256) unsigned char scratch[MX_STATIC_SCRATCH_BYTES];

namespace mx {

static thread_local char g_err[512] = "";

int set_error(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

namespace {

inline bool is_elem(int d) { return d == MX_E4M3 || d == MX_E5M2 || d == MX_E2M1; }
inline int64_t round256(int64_t b) { return (b + 255) & ~(int64_t)255; }

// kernel MX_KERNEL_AUTO uses for large problems
constexpr int big_tile_kernel() { return MX_KERNEL_MFMA_PINGPONG; }

// Problems with enough 256x256 tiles to occupy most of the 256 CUs are never split along K.
inline bool big_tile_problem(int64_t M, int64_t N) {
  return M > 128 && N > 128 && ((M + 255) / 256) * ((N + 255) / 256) >= 144;
}

// native scale layout a kernel reads: the two kernels on the 32x32x64 instruction have their own
inline int native_layout_of(int kernel) {
  return (kernel == MX_KERNEL_MFMA_PINGPONG32 || kernel == MX_KERNEL_MFMA_W4_PERSISTENT) ? MX_SCALE_NATIVE32
                                                                                       : MX_SCALE_NATIVE;
}
inline bool is_native(int layout) { return layout == MX_SCALE_NATIVE || layout == MX_SCALE_NATIVE32; }

// The decode kernel keeps X in registers: K up to kDecodeMaxK, 32 rows per launch (MX_KERNEL_AUTO gives it no more; an
// explicit MX_KERNEL_DECODE runs up to kDecodeMaxM rows slab by slab, each slab streaming the weights again).
constexpr int64_t kDecodeMaxK = 8192, kDecodeMaxM = 128;
// Rows up to which MX_KERNEL_AUTO streams the weights through registers (MX_KERNEL_STREAM).
constexpr int64_t kStreamAutoM = 64;
// FP4 weights with plain scales at up to 32 rows: the decode kernel keeps X in registers for the whole launch, which
// pays once a workgroup walks several weight tiles (28672 x 8192: 26 - 29 us against 28 - 36 us at 4 - 32 rows, 14336 x
// 4096 at 16 rows 11.4 against 10.9); beyond 16 rows, where X is as much as the weights, from the start, unless K is
// so short that its tiles are all start-up.
inline bool decode_beats_stream(int64_t M, int64_t N, int64_t K) {
  if (K > kDecodeMaxK || K % 512 != 0 || N % 16 != 0) return false;
  return M <= 16 ? (N >= 16384 && K >= 4096) : (K >= 2048 || N <= 8192);
}
const mx_gemm_opts kDefaultOpts = {sizeof(mx_gemm_opts), 0, MX_SCALE_2D, MX_SCALE_2D, MX_KERNEL_AUTO, 32, 0, 0};

// Number of K-slices for a problem that ends up on a one-tile MFMA kernel (1 = no split).  Depends only on
// (M, N, K, opts) so that mx_gemm_workspace_bytes and mx_gemm agree.  Automatic rule: split when the tiles
// of the 128x128 kernel cover less than half of the CUs and every slice keeps at least two K-quads.
int plan_k_splits(int64_t M, int64_t N, int64_t K, const mx_gemm_opts& o) {
  const bool t256 = o.kernel == MX_KERNEL_MFMA_256x256 || o.kernel == MX_KERNEL_MFMA_256x256_W4;
  if (o.split_k == 1 || o.block_size != 32 || K <= 0 || M <= 0 || N <= 0) return 1;
  if (o.kernel != MX_KERNEL_AUTO && o.kernel != MX_KERNEL_MFMA_128x128 && !t256) return 1;
  if (t256 && (o.a_scale_layout != MX_SCALE_2D || o.b_scale_layout != MX_SCALE_2D || K % 512 != 0)) return 1;
  if (o.split_k > 1) {   // -1: cannot honour; a K or scale layout that has never been split runs whole
    if (K % ((int64_t)512 * o.split_k) == 0) return o.split_k;
    return K % 512 == 0 && o.a_scale_layout == MX_SCALE_2D && o.b_scale_layout == MX_SCALE_2D ? -1 : 1;
  }
  if (t256) return 1;
  if (o.kernel == MX_KERNEL_AUTO && big_tile_problem(M, N)) return 1;   // big-tile kernel
  const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128);
  if (tiles * 2 > 256 || K < 2048) return 1;
  const int64_t s = 256 / tiles < K / 1024 ? 256 / tiles : K / 1024;
  return (int)(s < 1 ? 1 : s);
}


// What MX_KERNEL_AUTO weighs beyond kStreamAutoM rows: estimated time (us) of a product on the kernels that can run it.
// Fitted to measurements of 96 .. 4096 rows x 512 .. 28672 columns x 512 .. 9216 (stages of 128 bytes of a row, launches
// back to back, MXFP8; FP4 x FP4 has constants of its own):
//   64 x 64 and 128 x 128 tiles (mx_gemm_t128.hip picks by their number): a stage of 64 x 64 tiles 0.25 us with one on a CU
//     (1024 x 1024 x 4096 13.4 us), 0.42 with two (512 x 4096 x 4096 17.1, 335 x 2896 x 6144 24.3, x 12288 45.5), 0.21
//     and 0.32 with FP4 weights (221 x 4096 x 1408 6.7, 221 x 7424 x 1408 7.8, 200 x 8192 x 2048 9.4); of 128 x 128
//     ones 0.53 with one on every other CU (335 x 2896 x 12288 in two slices 36.5), 0.62 with one on each (2048 x 2048 x 8192
//     45), then by their number (2048 x 4096 x 4096 40, 1531 x 14336 x 4096 95).  Split along K: the partial sums are written
//     and read by a second launch (335 x 2896 x 6144 in 1, 2, 3, 6, 12 slices 24.3, 24.3, 21.5, 23.4, 32.3 us; 128 x 1024 x
//     12288 in 1, 4, 6, 12: 28.4, 15.7, 15.0, 17.2).
//   256 x 256 tiles: a round's length and, as the clock falls the busier the chip is, its share of tiles (4096^3, one full
//     round, 50; 2048 x 4096 x 4096, half of one, 44; 1531 x 14336 x 4096, 1.31 rounds, 86); it needs re-laid scales.
//   192 x 256 tiles: a round of them is 18 % shorter for 25 % fewer rows (more of a stage is not MFMA), which pays where it
//     fills rounds that 256 rows leave half empty (1531 x 14336 x 4096, 1.75 rounds, 77; 3000 x 4096 x 4096 42 against 45;
//     but 4096 x 14336 x 4096 187 against 175).
//   streaming: 0.5 .. 0.75 us per unit of its own cost estimate (64 x 4096 x 4096 9.4 us, 128 x 4096 x 8192 15.2, FP4 weights
//     12.1), or the time that reading the weights takes, longer the more row tiles share them (14336 x 8192, 64, 128, 256 rows:
//     28.6, 47, 83 us).  33 .. 64 rows: 64 x 64 tiles are faster for K up to 1024 (64 x 4096 x 1024 6.3 us against 7.8) and
//     for many columns (64 x 28672 x 2048 12.7 against 15.4), streaming for few and long ones (64 x 4096 x 4096 12.3 against 9.4).
float est_t128_split(int64_t M, int64_t N, int64_t K, int S, bool fp4, int64_t batch, bool fp4_b) {
  const int64_t small = t128_small_tiles(M, N) * S * batch, wgs = ((M + 127) / 128) * ((N + 127) / 128) * S * batch;
  const float st = (float)((K + (fp4 ? 255 : 127)) / (fp4 ? 256 : 128)) / S;
  float stage;
  if (small <= kT128SmallTiles) stage = small <= 256 ? (fp4 ? 0.33f : fp4_b ? 0.21f : 0.25f) : (fp4 ? 0.47f : fp4_b ? 0.32f : 0.42f);
  else if (wgs <= 256) stage = 0.42f + (fp4 ? 0.26f : 0.20f) * wgs / 256;
  else stage = 0.1f + (fp4 ? 1.25f : 1.05f) * (wgs < 435 ? 0.85f : wgs / 512.f);
  float t = 4.5f + st * stage;
  if (small <= kT128SmallTiles) {   // many columns for few rows: the time that reading B takes
    const float b = (float)N * K * (fp4_b ? 0.5f : 1.f) * batch;
    const float read = 1.3f + b / (b < 96e6f ? 4.8e6f : 3.8e6f);
    if (read > t) t = read;
  }
  return t + (S > 1 ? 3.f + 0.25f * S + (float)S * M * N * 8 / 5.5e6f : 0.f);
}
// Of the ways to split K that there is room for (up to S; automatic splits only) the best one: none, all, or as many as give
// every CU one or two 64 x 64 tiles.
int t128_splits(int64_t M, int64_t N, int64_t K, int S, bool fp4, bool fp4_b) {
  if (S <= 1) return 1;
  const int64_t w = t128_small_tiles(M, N);
  int best = 1;
  float us = est_t128_split(M, N, K, 1, fp4, 1, fp4_b);
  for (const int64_t s : {(int64_t)S, 256 / w, 512 / w}) {
    if (s < 2 || s > S) continue;
    const float t = est_t128_split(M, N, K, (int)s, fp4, 1, fp4_b);
    if (t < us) { us = t; best = (int)s; }
  }
  return best;
}
float est_t128(int64_t M, int64_t N, int64_t K, int S, bool fp4, bool fp4_b, int64_t batch = 1) {
  return est_t128_split(M, N, K, batch == 1 ? t128_splits(M, N, K, S, fp4, fp4_b) : 1, fp4, batch, fp4_b);
}
float est_pp(int64_t M, int64_t N, int64_t K, bool fp4, bool pack, bool tail, int rows = 256) {
  const int64_t tiles = ((M + rows - 1) / rows) * ((N + 255) / 256);
  const float st = (float)((K + (fp4 ? 255 : 127)) / (fp4 ? 256 : 128)), rest = 6.f + (pack ? 5.f : 0.f);
  const float round = rows == 256 ? (fp4 ? 1.14f : 0.95f) : (fp4 ? 0.80f : 0.79f), full = rows == 256 ? (fp4 ? 0.75f : 0.47f) : (fp4 ? 0.70f : 0.35f);
  if (tail) {   // the last round split S ways, its partial sums added up by a second launch
    const int left = (int)((tiles % 256 + 7) / 8), KQ = (int)(K / 512), S = tail_splits(left, 32, KQ, fp4);
    if (S > 1) return rest + st * (round + full) * (tiles / 256) + tail_tenths(S, left, 32, KQ, fp4) * 0.1f;
  }
  return rest + st * (round * ((tiles + 255) / 256) + full * tiles / 256);
}
// rows of the ping-pong kernel's tiles under MX_KERNEL_AUTO, and what they take; tail: there is room to split the last round of 256-row
// tiles (the 192-row form never splits)
struct PpRows { int rows; float us; };
PpRows pp_rows(int64_t M, int64_t N, int64_t K, bool fp4, bool pack, bool tail) {
  const float us = est_pp(M, N, K, fp4, pack, tail), us192 = est_pp(M, N, K, fp4, pack, false, 192);
  return us192 < us ? PpRows{192, us192} : PpRows{256, us};
}
float est_stream(int64_t M, int64_t N, int64_t K, int w_fmt) {
  const StreamPlan p = stream_plan(M, N, K, w_fmt);
  const bool fp4 = w_fmt == MX_E2M1;
  // (the plan's cost is that of its longest wave: where K-quads do not divide evenly, most waves are shorter)
  const int64_t KQ = (K + 511) / 512;
  const float rounds = (float)(((int64_t)p.units * p.m_tiles + 255) / 256) * 3.f;
  const float cost = rounds + (p.cost - rounds) * ((float)KQ / p.kw) / (float)((KQ + p.kw - 1) / p.kw);
  const float t = !fp4 ? 3.f + 0.55f * cost : p.mt == 4 ? 3.2f + 0.75f * cost : 2.6f + 0.5f * cost;
  const float read = 1.3f + (float)N * K * (fp4 ? 0.5f : 1.f) / 4.2e6f * (0.3f + 0.7f * p.m_tiles);
  return t > read ? t : read;
}

int check_tensor(const mx_tensor* t, const char* name, int min_nd, int max_nd) {
  if (!t) return set_error(MX_ERR_INVALID, "%s: null descriptor", name);
  if (t->ndim < min_nd || t->ndim > max_nd)
    return set_error(MX_ERR_SHAPE, "%s: expected %d..%d dimensions, got %d", name, min_nd, max_nd, t->ndim);
  int64_t numel = 1;
  for (int i = 0; i < t->ndim; ++i) {
    if (t->shape[i] < 0) return set_error(MX_ERR_SHAPE, "%s: negative extent", name);
    if (t->stride[i] < 0) return set_error(MX_ERR_LAYOUT, "%s: negative strides are not supported", name);
    numel *= t->shape[i];
  }
  if (numel > 0 && !t->ptr) return set_error(MX_ERR_INVALID, "%s: null data pointer", name);
  return MX_OK;
}

bool pair_supported_by_mfma(int a, int b) {
  return (a == MX_E4M3 && b == MX_E4M3) || (a == MX_E5M2 && b == MX_E5M2) ||
         (a == MX_E2M1 && b == MX_E2M1) || (a == MX_E4M3 && b == MX_E2M1);
}

// Checks the layout preconditions of the MFMA kernels for a K-contiguous operand with `rows` rows.
// Returns nullptr if fine, otherwise the reason.
const char* mfma_operand_issue(const void* ptr, int64_t rows, int64_t K, int64_t ld_bytes, int64_t k_stride,
                               int fmt, int packed_ok) {
  if (k_stride != 1) return "K axis is not contiguous";
  if (fmt == MX_E2M1 && !packed_ok) return "FP4 operand is not packed along K";
  if (((uintptr_t)ptr) % 16 != 0) return "base pointer is not 16-byte aligned";
  if (ld_bytes % 16 != 0) return "row pitch is not a multiple of 16 bytes";
  const int64_t row = fmt == MX_E2M1 ? K / 2 : K, lim = (int64_t)1 << 31;
  if (rows * ld_bytes >= lim || (rows - 1) * ld_bytes + row >= lim) return "operand spans 2 GiB or more";   // (rows may overlap)
  return nullptr;
}

constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

// device address of `scratch` on the current device (each GPU holds its own copy at its own address)
int static_scratch(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return set_error(MX_ERR_DEVICE, "hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return set_error(MX_ERR_DEVICE, "device index %d out of range", dev);
  void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!p) {
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return set_error(MX_ERR_DEVICE, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    g_scratch_ptr[dev].store(p, std::memory_order_release);   // a racing thread stores the same address
  }
  *out = p;
  return MX_OK;
}
}  // namespace
}  // namespace mx

using namespace mx;

extern "C" {

int mx_version(void) { return MXGEMM_VERSION; }

const char* mx_last_error(void) { return g_err; }

int mx_device_check(void) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return set_error(MX_ERR_DEVICE, "hipGetDevice: %s", hipGetErrorString(e));
  hipDeviceProp_t prop;
  e = hipGetDeviceProperties(&prop, dev);
  if (e != hipSuccess) return set_error(MX_ERR_DEVICE, "hipGetDeviceProperties: %s", hipGetErrorString(e));
  if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return set_error(MX_ERR_DEVICE, "libmxgemm is built for gfx950 only, device is %s", prop.gcnArchName);
  void* p = nullptr;
  return static_scratch(&p);   // set-up of mx_gemm_static on this device
}

int64_t mx_packed_scale_bytes(int64_t rows, int64_t K) {
  return round256(packed_scale_dwords(rows, K) * 4);
}

namespace {
// re-laid scales, partial sums of split-K
int64_t gemm_workspace_min(int64_t M, int64_t N, int64_t K, const mx_gemm_opts& o) {
  if (o.kernel == MX_KERNEL_GENERIC || o.kernel == MX_KERNEL_STREAM || o.kernel == MX_KERNEL_DECODE) return 0;
  int64_t b = 0;
  const int S = plan_k_splits(M, N, K, o);
  if (S > 1) b += round256(S * M * N * 4);   // the fp32 partial products
  if (!is_native(o.a_scale_layout)) b += mx_packed_scale_bytes(M, K);
  if (!is_native(o.b_scale_layout)) b += mx_packed_scale_bytes(N, K);
  return b;
}
// Partial sums that a caller is held to: of a split into equal slices of 512 with plain scales, as mx_gemm_opts::split_k has it
// (an automatic one: the most such slices within it).  Every other split is the library's own choice; where its partial
// sums have no room the product runs whole.
int64_t held_partial_sums(int64_t M, int64_t N, int64_t K, const mx_gemm_opts& o) {
  if (K % 512 != 0 || o.a_scale_layout != MX_SCALE_2D || o.b_scale_layout != MX_SCALE_2D) return 0;
  int S = plan_k_splits(M, N, K, o);
  while (S > 1 && K % ((int64_t)512 * S) != 0) --S;
  return S > 1 ? round256((int64_t)S * M * N * 4) : 0;
}
// what mx_gemm cannot do without, and the options that a product runs under with `bytes` of workspace
int64_t gemm_workspace_held(int64_t M, int64_t N, int64_t K, const mx_gemm_opts& o) {
  mx_gemm_opts whole = o;
  whole.split_k = 1;
  return gemm_workspace_min(M, N, K, whole) + held_partial_sums(M, N, K, o);
}
mx_gemm_opts opts_for_room(int64_t M, int64_t N, int64_t K, const mx_gemm_opts& o, int64_t bytes) {
  mx_gemm_opts r = o;
  if (bytes < gemm_workspace_min(M, N, K, o) && bytes >= gemm_workspace_held(M, N, K, o)) r.split_k = 1;
  return r;
}
// beyond that, what lets the ping-pong kernel split its last round along K (0: it would not): only for problems that it may
// be picked for
int64_t gemm_workspace_tail(int64_t M, int64_t N, int64_t K, const mx_gemm_opts& o) {
  if ((o.kernel != MX_KERNEL_AUTO && o.kernel != MX_KERNEL_MFMA_PINGPONG) || o.split_k != 0 || o.block_size != 32 || M <= 0 || N <= 0 ||
      K <= 0)
    return 0;
  const int64_t t = pp_tail_bytes(M, N, K, false, true);
  if (t == 0 || o.kernel == MX_KERNEL_MFMA_PINGPONG) return t;
  if (M <= kStreamAutoM) return 0;
  const bool pack = !is_native(o.a_scale_layout) || !is_native(o.b_scale_layout);
  for (int fp4 = 0; fp4 < 2; ++fp4) {
    const PpRows with = pp_rows(M, N, K, fp4, pack, true);
    // (192 rows with room and without it: nothing is split)
    if (with.rows == 192 && pp_rows(M, N, K, fp4, pack, false).rows == 192) continue;
    if (with.us < est_t128(M, N, K, plan_k_splits(M, N, K, o), fp4, fp4)) return t;
  }
  return 0;
}
int64_t grouped_workspace_min(int64_t num_slots, int64_t N, int64_t K, int64_t E, const mx_gemm_opts& o) {
  if (o.kernel == MX_KERNEL_GENERIC) return 0;
  int64_t b = mx_packed_scale_bytes(num_slots, K);
  if (!is_native(o.b_scale_layout)) b += E * mx_packed_scale_bytes(N, K);
  return b;
}
}  // namespace

int64_t mx_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K, const mx_gemm_opts* opts) {
  const mx_gemm_opts& o = opts ? *opts : kDefaultOpts;
  return gemm_workspace_min(M, N, K, o) + gemm_workspace_tail(M, N, K, o);
}

int64_t mx_gemm_grouped_workspace_bytes(int64_t num_slots, int64_t N, int64_t K, int64_t E,
                                        const mx_gemm_opts* opts) {
  const mx_gemm_opts& o = opts ? *opts : kDefaultOpts;
  const bool pp = (o.kernel == MX_KERNEL_AUTO && N > 128) || o.kernel == MX_KERNEL_MFMA_PINGPONG;
  return grouped_workspace_min(num_slots, N, K, E, o) + (pp ? pp_tail_bytes(num_slots, N, K, false, false) : 0);
}

namespace {
// a 4-D swizzle_32_4_4 scale tensor must be the contiguous [rows / 128, (K / 32) / 4, 32, 16] array
int check_swizzled_scale(const mx_tensor* scale, const char* name, int64_t rows, int64_t KB) {
  if (scale->ndim != 4 || scale->shape[2] != 32 || scale->shape[3] != 16)
    return set_error(MX_ERR_SHAPE, "%s: swizzled scale layout expects [rows/128, K/128, 32, 16]", name);
  if (rows % 128 != 0 || KB % 4 != 0 || scale->shape[0] != rows / 128 || scale->shape[1] != KB / 4)
    return set_error(MX_ERR_SHAPE, "%s: swizzled scale shape does not match rows=%lld, K blocks=%lld (rows %% 128 "
                     "and blocks %% 4 must be 0)", name, (long long)rows, (long long)KB);
  if (scale->stride[3] != 1 || scale->stride[2] != 16 || scale->stride[1] != 512 ||
      scale->stride[0] != 512 * (KB / 4))
    return set_error(MX_ERR_LAYOUT, "%s: swizzled scale tensor must be contiguous", name);
  return MX_OK;
}

// validates a scale tensor against (rows, K) and describes its re-layout into `packed`
int make_pack_args(const mx_tensor* scale, int32_t layout, int64_t rows, int64_t K, void* packed, int target,
                   PackArgs& p) {
  if (int rc = check_tensor(scale, "scale", 2, 4)) return rc;
  if (!packed) return set_error(MX_ERR_INVALID, "packed: null pointer");
  if (K % 32 != 0) return set_error(MX_ERR_SHAPE, "K (%lld) must be a multiple of 32", (long long)K);
  if (((uintptr_t)packed) % 16 != 0) return set_error(MX_ERR_LAYOUT, "packed buffer must be 16-byte aligned");
  p = PackArgs{};
  p.src = (const uint8_t*)scale->ptr;
  p.dst = (uint32_t*)packed;
  p.rows = rows;
  p.K = K;
  p.layout = layout;
  p.target = target;
  p.batch = 1;
  p.replicas = 1;
  const int64_t KB = K / 32;
  if (layout == MX_SCALE_2D) {
    const int nd = scale->ndim;
    if (nd != 2 && nd != 3) return set_error(MX_ERR_SHAPE, "2-D scale layout expects [rows, K/32] with an optional batch");
    if (scale->shape[nd - 2] != rows || scale->shape[nd - 1] != KB)
      return set_error(MX_ERR_SHAPE, "scale shape (%lld, %lld) does not match rows=%lld, K/32=%lld",
                       (long long)scale->shape[nd - 2], (long long)scale->shape[nd - 1], (long long)rows,
                       (long long)KB);
    p.s_row = scale->stride[nd - 2];
    p.s_kb = scale->stride[nd - 1];
    if (nd == 3) {
      p.batch = (int32_t)scale->shape[0];
      p.s_batch = scale->stride[0];
    }
  } else if (layout == MX_SCALE_SWIZZLE_32_4_4) {
    if (int rc = check_swizzled_scale(scale, "scale", rows, KB)) return rc;
  } else {
    return set_error(MX_ERR_INVALID, "mx_pack_scales: unknown source layout %d", layout);
  }
  return MX_OK;
}
}  // namespace

int mx_pack_scales(const mx_tensor* scale, int32_t layout, int64_t rows, int64_t K, int32_t native_layout,
                   int32_t operand, void* packed, void* stream) {
  if (!is_native(native_layout))
    return set_error(MX_ERR_INVALID, "mx_pack_scales: native_layout must be MX_SCALE_NATIVE or MX_SCALE_NATIVE32");
  if (operand != MX_OPERAND_A && operand != MX_OPERAND_B)
    return set_error(MX_ERR_INVALID, "mx_pack_scales: operand must be MX_OPERAND_A or MX_OPERAND_B");
  const int target = native_layout == MX_SCALE_NATIVE32 ? kPackTile32 : (operand == MX_OPERAND_B ? kPackB : kPackA);
  PackArgs p;
  if (int rc = make_pack_args(scale, layout, rows, K, packed, target, p)) return rc;
  return launch_pack_scales(p, (hipStream_t)stream);
}

namespace {
// What mx_gemm would launch for a problem that ends on the 128 x 128 one-tile kernel without split-K: the list
// entry point collects these and runs them as one batched scale re-layout and one persistent GEMM launch.
struct GemmPlan {
  T128Args g;
  PackArgs pa, pb;
  bool pack_a, pack_b;
};
constexpr int kPlanNotSimple = 1;   // gemm_impl with a plan: the problem needs its own mx_gemm call
constexpr int kAccNeedsCopy = 2;    // gemm_impl with an addend: the kernel can only accumulate into C (nothing enqueued)

int gemm_impl(const mx_tensor* A, const mx_tensor* As, const mx_tensor* B, const mx_tensor* Bs, mx_tensor* C,
              const mx_gemm_opts* opts, void* workspace, int64_t workspace_bytes, void* stream, GemmPlan* plan,
              const float* acc = nullptr);
}  // namespace

int mx_gemm(const mx_tensor* A, const mx_tensor* As, const mx_tensor* B, const mx_tensor* Bs, mx_tensor* C,
            const mx_gemm_opts* opts, void* workspace, int64_t workspace_bytes, void* stream) {
  return gemm_impl(A, As, B, Bs, C, opts, workspace, workspace_bytes, stream, nullptr);
}

int mx_gemm_add(const mx_tensor* A, const mx_tensor* As, const mx_tensor* B, const mx_tensor* Bs, const mx_tensor* D,
                mx_tensor* C, const mx_gemm_opts* opts, void* workspace, int64_t workspace_bytes, void* stream) {
  if (int rc = check_tensor(D, "D", 2, 3)) return rc;
  if (int rc = check_tensor(C, "C", 2, 3)) return rc;
  if (D->dtype != MX_F32 || C->dtype != MX_F32) return set_error(MX_ERR_DTYPE, "mx_gemm_add: D and C must be MX_F32");
  if (D->ndim != C->ndim) return set_error(MX_ERR_SHAPE, "mx_gemm_add: D and C must have the same shape");
  int64_t numel = 1;
  for (int i = C->ndim - 1; i >= 0; --i) {
    if (D->shape[i] != C->shape[i]) return set_error(MX_ERR_SHAPE, "mx_gemm_add: D and C must have the same shape");
    if (C->shape[i] > 1 && (D->stride[i] != numel || C->stride[i] != numel))
      return set_error(MX_ERR_LAYOUT, "mx_gemm_add: D and C must be contiguous");
    numel *= C->shape[i];
  }
  mx_gemm_opts o = opts ? *opts : kDefaultOpts;
  o.accumulate = 0;
  const int rc = gemm_impl(A, As, B, Bs, C, &o, workspace, workspace_bytes, stream, nullptr, (const float*)D->ptr);
  if (rc != kAccNeedsCopy) return rc;
  if (numel == 0) return MX_OK;
  if (C->ptr != D->ptr) {
    const hipError_t e = hipMemcpyAsync(C->ptr, D->ptr, (size_t)numel * 4, hipMemcpyDeviceToDevice, (hipStream_t)stream);
    if (e != hipSuccess) return set_error(MX_ERR_DEVICE, "mx_gemm_add: %s", hipGetErrorString(e));
  }
  o.accumulate = 1;
  return gemm_impl(A, As, B, Bs, C, &o, workspace, workspace_bytes, stream, nullptr);
}

namespace {
// mx_gemm; with `plan` nothing is launched: a problem of the simple kind is described in *plan (return MX_OK),
// any other valid problem returns kPlanNotSimple.  acc: fp32 addend laid out like C (contiguous)
int gemm_impl(const mx_tensor* A, const mx_tensor* As, const mx_tensor* B, const mx_tensor* Bs, mx_tensor* C,
              const mx_gemm_opts* opts, void* workspace, int64_t workspace_bytes, void* stream, GemmPlan* plan,
              const float* acc) {
  mx_gemm_opts o = opts ? *opts : kDefaultOpts;
  if (int rc = check_tensor(A, "A", 2, 3)) return rc;
  if (int rc = check_tensor(B, "B", 2, 3)) return rc;
  if (int rc = check_tensor(As, "A_scale", 2, 4)) return rc;
  if (int rc = check_tensor(Bs, "B_scale", 2, 4)) return rc;
  if (int rc = check_tensor(C, "C", 2, 3)) return rc;
  if (!is_elem(A->dtype) || !is_elem(B->dtype))
    return set_error(MX_ERR_DTYPE, "A/B must be MX_E4M3, MX_E5M2 or MX_E2M1 (got %d, %d)", A->dtype, B->dtype);
  if (C->dtype != MX_F32 && C->dtype != MX_BF16)
    return set_error(MX_ERR_DTYPE, "C must be MX_F32 or MX_BF16 (got %d)", C->dtype);
  if (As->dtype != Bs->dtype) return set_error(MX_ERR_DTYPE, "A_scale and B_scale must have the same dtype");
  if (As->dtype != MX_E8M0 && As->dtype != MX_E4M3)
    return set_error(MX_ERR_DTYPE, "scale dtype must be MX_E8M0 (or MX_E4M3 for FP4 with block 16)");
  if (o.block_size != 32 && o.block_size != 16)
    return set_error(MX_ERR_INVALID, "block_size must be 16 or 32 (got %d)", o.block_size);

  const int and_ = A->ndim, bnd = B->ndim, cnd = C->ndim;
  const int64_t M = A->shape[and_ - 2], K = A->shape[and_ - 1];
  const int64_t Kb = B->shape[bnd - 2], N = B->shape[bnd - 1];
  if (K != Kb)
    return set_error(MX_ERR_SHAPE, "Incompatible matrices: K dimension of A (%lld) must match K dimension of B (%lld)",
                     (long long)K, (long long)Kb);
  if (K % o.block_size != 0)
    return set_error(MX_ERR_SHAPE, "K (%lld) must be a multiple of the scaling block size %d", (long long)K,
                     o.block_size);
  const int64_t batchA = and_ == 3 ? A->shape[0] : 1, batchB = bnd == 3 ? B->shape[0] : 1;
  if (batchA != batchB && batchA != 1 && batchB != 1)
    return set_error(MX_ERR_SHAPE, "batch dimensions %lld and %lld cannot be broadcast", (long long)batchA,
                     (long long)batchB);
  const int64_t batch = batchA > batchB ? batchA : batchB;
  const bool batched = and_ == 3 || bnd == 3;
  if ((batched && (cnd != 3 || C->shape[0] != batch)) || (!batched && cnd != 2) || C->shape[cnd - 2] != M ||
      C->shape[cnd - 1] != N)
    return set_error(MX_ERR_SHAPE, "C has the wrong shape for a (%lld x %lld x %lld) product", (long long)M,
                     (long long)N, (long long)K);
  if (A->dtype == MX_E2M1 && A->packed_dim != and_ - 1 && A->packed_dim != and_ - 2)
    return set_error(MX_ERR_LAYOUT, "A: packed_dim must name the M or K dimension");
  if (B->dtype == MX_E2M1 && B->packed_dim != bnd - 1 && B->packed_dim != bnd - 2)
    return set_error(MX_ERR_LAYOUT, "B: packed_dim must name the K or N dimension");
  const int64_t KB = K / o.block_size;

  // ---- scale shapes --------------------------------------------------------------------------------
  if (o.a_scale_layout == MX_SCALE_2D) {
    const int nd = As->ndim;
    if (nd != and_ || As->shape[nd - 2] != M || As->shape[nd - 1] != KB || (nd == 3 && As->shape[0] != batchA))
      return set_error(MX_ERR_SHAPE, "A_scale shape is not compatible with A: expected [.., %lld, %lld]",
                       (long long)M, (long long)KB);
  }
  if (o.b_scale_layout == MX_SCALE_2D) {
    const int nd = Bs->ndim;
    if (nd != bnd || Bs->shape[nd - 2] != KB || Bs->shape[nd - 1] != N || (nd == 3 && Bs->shape[0] != batchB))
      return set_error(MX_ERR_SHAPE, "B_scale shape is not compatible with B: expected [.., %lld, %lld]",
                       (long long)KB, (long long)N);
  }
  if (M == 0 || N == 0) return plan ? kPlanNotSimple : MX_OK;

  // ---- batched operands (test/test_mma_scaled.py:128-145): one 2-D product per batch entry, size-1
  // batches broadcast; stream order lets the entries share the workspace.  Layouts only the generic
  // kernel reads (block 16, E4M3 scales) keep its own batched launch. --------------------------------
  if (batched && o.kernel != MX_KERNEL_GENERIC && o.block_size == 32 && As->dtype == MX_E8M0 &&
      o.a_scale_layout == MX_SCALE_2D && o.b_scale_layout == MX_SCALE_2D) {
    if (plan) return kPlanNotSimple;
    auto slice = [](const mx_tensor* t, int64_t b, int elem_bytes) {
      mx_tensor v = *t;
      if (t->ndim == 3) {
        v.ptr = (uint8_t*)t->ptr + (t->shape[0] > 1 ? b : 0) * t->stride[0] * elem_bytes;
        v.ndim = 2;
        for (int i = 0; i < 2; ++i) { v.shape[i] = t->shape[i + 1]; v.stride[i] = t->stride[i + 1]; }
        if (v.packed_dim >= 0) v.packed_dim -= 1;
      }
      return v;
    };
    // small products: the whole batch as one launch of the 128 x 128 kernel (behind one scale re-layout launch), in chunks
    // of what the workspace holds packed scales for
    {
      const mx_tensor a2 = slice(A, 0, 1), b2 = slice(B, 0, 1), as2 = slice(As, 0, 1), bs2 = slice(Bs, 0, 1);
      auto bstride = [](const mx_tensor* t) { return t->ndim == 3 && t->shape[0] > 1 ? t->stride[0] : (int64_t)0; };
      const int64_t per = mx_packed_scale_bytes(M, K) + mx_packed_scale_bytes(N, K);
      const bool fp4 = A->dtype == MX_E2M1;
      bool ok = (o.kernel == MX_KERNEL_AUTO || o.kernel == MX_KERNEL_MFMA_128x128) && o.split_k <= 1 && K > 0 &&
                pair_supported_by_mfma(A->dtype, B->dtype) && C->stride[2] == 1 && bstride(A) % 16 == 0 && bstride(B) % 16 == 0 &&
                !mfma_operand_issue(a2.ptr, M, K, a2.stride[0], a2.stride[1], A->dtype, a2.packed_dim == 1) &&
                !mfma_operand_issue(b2.ptr, N, K, b2.stride[1], b2.stride[0], B->dtype, b2.packed_dim == 0) &&
                M < (1 << 30) && N < (1 << 30) && K < (1 << 30);
      const bool plain = ok && t128_plain_scales(as2.ptr, as2.stride[0], as2.stride[1], M, K, A->dtype, B->dtype) &&
                         t128_plain_scales(bs2.ptr, bs2.stride[1], bs2.stride[0], N, K, A->dtype, B->dtype) &&
                         bstride(As) % 4 == 0 && bstride(Bs) % 4 == 0;
      const bool any = ok && !plain && t128_any_pays(M, N, K, batch, A->dtype == MX_E2M1 && B->dtype == MX_E2M1) &&
                       t128_any_scales(as2.stride[0], as2.stride[1], M, K) && t128_any_scales(bs2.stride[1], bs2.stride[0], N, K);
      int64_t chunk = plain ? batch : (workspace ? workspace_bytes / per : 0);
      if (any && chunk >= 1) chunk = batch;   // (reads the scales where they are; callers are held to the workspace all the same)
      if (chunk > 32768) chunk = 32768;
      if (ok && batch > 1) {   // few long products are better off one by one with K split, large ones gain nothing
        float alone = est_t128(M, N, K, plan_k_splits(M, N, K, o), fp4, B->dtype == MX_E2M1);
        if (o.kernel == MX_KERNEL_AUTO) {
          const float pp = est_pp(M, N, K, fp4, true, false);
          if (pp < alone) alone = pp;
          if (!fp4 && M <= kStreamAutoM && est_stream(M, N, K, B->dtype) < alone) alone = est_stream(M, N, K, B->dtype);
        }
        ok = est_t128(M, N, K, 1, fp4, B->dtype == MX_E2M1, batch) <= batch * alone;
      }
      if (!plain && workspace && ((uintptr_t)workspace) % 256 != 0) ok = false;
      if (ok && chunk >= 1) {
        for (int64_t b0 = 0; b0 < batch; b0 += chunk) {
          const int64_t nb = batch - b0 < chunk ? batch - b0 : chunk;
          T128Args g = {};
          g.A = (const uint8_t*)A->ptr + b0 * bstride(A); g.a_batch = bstride(A);
          g.B = (const uint8_t*)B->ptr + b0 * bstride(B); g.b_batch = bstride(B);
          g.As = (const uint8_t*)As->ptr + b0 * bstride(As); g.as_batch = bstride(As);
          g.Bs = (const uint8_t*)Bs->ptr + b0 * bstride(Bs); g.bs_batch = bstride(Bs);
          g.c_batch = C->stride[0];
          g.C = (uint8_t*)C->ptr + b0 * g.c_batch * (C->dtype == MX_BF16 ? 2 : 4);
          if (acc) g.acc = acc + b0 * g.c_batch;
          g.lda = a2.stride[0]; g.ldb = b2.stride[1]; g.ldas = as2.stride[0]; g.ldbs = bs2.stride[1]; g.ldc = C->stride[1];
          g.M = (int32_t)M; g.N = (int32_t)N; g.K = (int32_t)K;
          g.a_fmt = A->dtype; g.b_fmt = B->dtype; g.c_dtype = C->dtype; g.accumulate = o.accumulate;
          g.a_plain = g.b_plain = plain ? 1 : any ? kT128ScalesAny : 0;
          g.batch = (int32_t)nb; g.k_splits = 1; g.a_rows = M;
          if (!g.a_plain) {
            PackArgs pa, pb;
            mx_tensor t = bs2;
            t.shape[0] = bs2.shape[1]; t.shape[1] = bs2.shape[0];
            t.stride[0] = bs2.stride[1]; t.stride[1] = bs2.stride[0];
            uint8_t* const wa = (uint8_t*)workspace;
            const int64_t na = g.as_batch ? nb : 1, nbb = g.bs_batch ? nb : 1;   // a broadcast operand is re-laid once
            uint8_t* const wb = wa + na * mx_packed_scale_bytes(M, K);
            if (int rc = make_pack_args(&as2, MX_SCALE_2D, M, K, wa, kPackA, pa)) return rc;
            if (int rc = make_pack_args(&t, MX_SCALE_2D, N, K, wb, kPackB, pb)) return rc;
            pa.src = g.As; pa.batch = (int32_t)na; pa.s_batch = g.as_batch;
            pb.src = g.Bs; pb.batch = (int32_t)nbb; pb.s_batch = g.bs_batch;
            if (int rc = launch_pack_scales_pair(&pa, &pb, (hipStream_t)stream)) return rc;
            g.As = wa; g.Bs = wb;
            g.as_batch = g.as_batch ? mx_packed_scale_bytes(M, K) : 0;
            g.bs_batch = g.bs_batch ? mx_packed_scale_bytes(N, K) : 0;
          }
          if (int rc = launch_gemm_t128(g, (hipStream_t)stream)) return rc;
        }
        return MX_OK;
      }
    }
    if (acc) return kAccNeedsCopy;
    const int c_bytes = C->dtype == MX_BF16 ? 2 : 4;
    for (int64_t b = 0; b < batch; ++b) {
      const mx_tensor a2 = slice(A, b, 1), as2 = slice(As, b, 1), b2 = slice(B, b, 1), bs2 = slice(Bs, b, 1);
      mx_tensor c2 = slice(C, b, c_bytes);
      if (int rc = mx_gemm(&a2, &as2, &b2, &bs2, &c2, &o, workspace, workspace_bytes, stream)) return rc;
    }
    return MX_OK;
  }

  int64_t ws_min = batched ? 0 : gemm_workspace_min(M, N, K, o);
  if (ws_min > (workspace ? workspace_bytes : 0)) {
    o = opts_for_room(M, N, K, o, workspace ? workspace_bytes : 0);
    ws_min = gemm_workspace_min(M, N, K, o);
  }
  // ---- can the MFMA path take it? ------------------------------------------------------------------
  const char* why = nullptr;
  const int64_t a_ld = A->stride[and_ - 2], b_ld = B->stride[bnd - 1];
  if (batched) why = "batched operands";
  else if (o.block_size != 32 || As->dtype != MX_E8M0) why = "only E8M0 scales with block 32 are MFMA-native";
  else if (!pair_supported_by_mfma(A->dtype, B->dtype)) why = "element format pair not instantiated";
  else if (K == 0) why = "K is zero";
  else if ((why = mfma_operand_issue(A->ptr, M, K, a_ld, A->stride[1], A->dtype, A->packed_dim == 1))) {}
  else if ((why = mfma_operand_issue(B->ptr, N, K, b_ld, B->stride[0], B->dtype, B->packed_dim == 0))) {}
  else if (C->stride[1] != 1) why = "C is not row-major";
  else if (M >= (1 << 30) || N >= (1 << 30) || K >= (1 << 30)) why = "extent too large";

  // what keeps the weight-streaming kernel from taking the problem (it also takes E5M2 x E2M1, which the tiled
  // kernels do not)
  StreamArgs sa = {};
  const char* why_stream = nullptr;
  if (batched) why_stream = "batched operands";
  else if (o.block_size != 32 || As->dtype != MX_E8M0) why_stream = "it reads E8M0 scales with block 32";
  else if (M >= (1 << 30) || N >= (1 << 30) || K >= (1 << 30)) why_stream = "extent too large";
  else if (A->stride[1] != 1 || B->stride[0] != 1) why_stream = "K axis is not contiguous";
  else if (B->dtype == MX_E2M1 && B->packed_dim != 0) why_stream = "FP4 operand is not packed along K";
  else if (C->stride[1] != 1) why_stream = "C is not row-major";
  else if (o.a_scale_layout != MX_SCALE_2D || As->stride[1] != 1) why_stream = "A_scale must be the plain K-contiguous layout";
  else if (o.b_scale_layout != MX_SCALE_NATIVE && (o.b_scale_layout != MX_SCALE_2D || Bs->stride[0] != 1))
    why_stream = "B_scale must be MX_SCALE_NATIVE or plain and K-contiguous";
  else {
    sa.X = (const uint8_t*)A->ptr; sa.Xs = (const uint8_t*)As->ptr;
    sa.W = (const uint8_t*)B->ptr; sa.Ws = (const uint8_t*)Bs->ptr; sa.C = C->ptr;
    sa.M = (int32_t)M; sa.N = (int32_t)N; sa.K = (int32_t)K;
    sa.ldx = a_ld; sa.ldxs = As->stride[0]; sa.ldw = b_ld; sa.ldws = Bs->stride[1]; sa.ldc = C->stride[0];
    sa.x_fmt = A->dtype; sa.w_fmt = B->dtype; sa.c_dtype = C->dtype; sa.accumulate = o.accumulate;
    sa.ws_packed = o.b_scale_layout == MX_SCALE_NATIVE;
    why_stream = stream_issue(sa);
  }

  int kernel = o.kernel, tile_rows = 256;
  if (kernel == MX_KERNEL_DECODE && K > kDecodeMaxK && M <= kDecodeMaxM && N % 16 == 0 && K % 512 == 0 && !why_stream &&
      o.b_scale_layout == MX_SCALE_2D && B->dtype == MX_E2M1)
    kernel = MX_KERNEL_STREAM;   // beyond what the decode kernel keeps of X in registers
  if (kernel == MX_KERNEL_STREAM) {
    if (why_stream) return set_error(MX_ERR_LAYOUT, "the streaming kernel cannot run this problem: %s", why_stream);
  } else if (kernel == MX_KERNEL_AUTO) {
    const bool may_stream = !plan && !why_stream && o.split_k <= 1;
    // (a call that would need the workspace on the tiled kernel and has none streams as it always did)
    const bool tiles = may_stream && !why && M > 32 && M <= kStreamAutoM && (ws_min == 0 || (workspace && workspace_bytes >= ws_min && ((uintptr_t)workspace) % 256 == 0)) &&
                       est_t128(M, N, K, plan_k_splits(M, N, K, o), A->dtype == MX_E2M1, B->dtype == MX_E2M1) <
                           est_stream(M, N, K, B->dtype);
    if (may_stream && (why || (M <= kStreamAutoM && !tiles)) &&
        !(M <= 32 && decode_beats_stream(M, N, K) && B->dtype == MX_E2M1 && o.b_scale_layout == MX_SCALE_2D))
      kernel = MX_KERNEL_STREAM;
    else if (why) kernel = MX_KERNEL_GENERIC;
    // (a longer K streams; here that is a problem of a list, which then gets a call of its own)
    else if (M <= 32 && (K <= kDecodeMaxK || !why_stream) && o.split_k <= 1 && A->dtype != MX_E2M1 && B->dtype == MX_E2M1 &&
             o.a_scale_layout == MX_SCALE_2D &&
             o.b_scale_layout == MX_SCALE_2D && Bs->stride[0] == 1 && As->stride[1] == 1 && K % 512 == 0 &&
             N % 16 == 0 && Bs->stride[1] % 16 == 0 && ((uintptr_t)Bs->ptr) % 16 == 0 &&
             N * b_ld < ((int64_t)1 << 31) && As->stride[0] % 16 == 0 && ((uintptr_t)As->ptr) % 16 == 0)
      kernel = MX_KERNEL_DECODE;
    else {
      const bool fp4 = A->dtype == MX_E2M1;
      const float t128 = est_t128(M, N, K, o.split_k > 1 ? 1 : plan_k_splits(M, N, K, o), fp4, B->dtype == MX_E2M1);
      const bool room = workspace && o.split_k == 0 && pp_tail_bytes(M, N, K, fp4, true) > 0 &&
                        workspace_bytes >= ws_min + pp_tail_bytes(M, N, K, fp4, true);
      const PpRows p = pp_rows(M, N, K, fp4, !is_native(o.a_scale_layout) || !is_native(o.b_scale_layout), room);
      const float pp = o.split_k > 1 ? 1e30f : p.us;
      if (o.split_k <= 1) tile_rows = p.rows;
      const float st = may_stream ? est_stream(M, N, K, B->dtype) : 1e30f;
      kernel = st < t128 && st < pp ? MX_KERNEL_STREAM : t128 <= pp ? MX_KERNEL_MFMA_128x128 : big_tile_kernel();
    }
  } else if (kernel != MX_KERNEL_GENERIC && why) {
    return set_error(MX_ERR_LAYOUT, "requested kernel %d cannot run this problem: %s", kernel, why);
  }

  if (o.split_k > 1 && kernel != MX_KERNEL_MFMA_128x128 && kernel != MX_KERNEL_MFMA_256x256 &&
      kernel != MX_KERNEL_MFMA_256x256_W4)
    return set_error(MX_ERR_LAYOUT, "split_k = %d is only available on the one-tile MFMA kernels (kernel %d chosen)",
                     o.split_k, kernel);
  if (plan && kernel != MX_KERNEL_MFMA_128x128) return kPlanNotSimple;
  if (acc && kernel != MX_KERNEL_MFMA_128x128) return kAccNeedsCopy;
  if (kernel == MX_KERNEL_GENERIC) {
    if (is_native(o.a_scale_layout) || is_native(o.b_scale_layout))
      return set_error(MX_ERR_LAYOUT, "the generic kernel cannot read native-layout scales");
    if (As->dtype == MX_E4M3 && !(A->dtype == MX_E2M1 && o.block_size == 16))
      return set_error(MX_ERR_DTYPE, "E4M3 scales are only defined for FP4 operands with block size 16");
    if (o.block_size == 16 && (A->dtype != MX_E2M1 || B->dtype != MX_E2M1))
      return set_error(MX_ERR_DTYPE, "block size 16 is only defined for FP4 operands");
    if (M > 0x7FFFFFFF || N > 0x7FFFFFFF || K > 0x7FFFFFFF || batch > 0x7FFFFFFF)
      return set_error(MX_ERR_SHAPE, "extents of 2^31 or more are not supported");
    if ((o.a_scale_layout == MX_SCALE_SWIZZLE_32_4_4 || o.b_scale_layout == MX_SCALE_SWIZZLE_32_4_4) && batched)
      return set_error(MX_ERR_LAYOUT, "swizzled scale tensors have no batch dimension");
    if (o.a_scale_layout == MX_SCALE_SWIZZLE_32_4_4)
      if (int rc = check_swizzled_scale(As, "A_scale", M, KB)) return rc;
    if (o.b_scale_layout == MX_SCALE_SWIZZLE_32_4_4)
      if (int rc = check_swizzled_scale(Bs, "B_scale", N, KB)) return rc;
    GenericArgs g = {};
    g.A = (const uint8_t*)A->ptr; g.As = (const uint8_t*)As->ptr;
    g.B = (const uint8_t*)B->ptr; g.Bs = (const uint8_t*)Bs->ptr; g.C = C->ptr;
    g.batch = (int32_t)batch; g.M = (int32_t)M; g.N = (int32_t)N; g.K = (int32_t)K; g.block = o.block_size;
    g.a_fmt = A->dtype; g.b_fmt = B->dtype; g.scale_fmt = As->dtype; g.c_dtype = C->dtype;
    g.accumulate = o.accumulate;
    g.a_packed_k = A->packed_dim == and_ - 1; g.b_packed_k = B->packed_dim == bnd - 2;
    g.a_sb = (and_ == 3 && batchA > 1) ? A->stride[0] : 0;
    g.a_sm = A->stride[and_ - 2]; g.a_sk = A->stride[and_ - 1];
    g.b_sb = (bnd == 3 && batchB > 1) ? B->stride[0] : 0;
    g.b_sk = B->stride[bnd - 2]; g.b_sn = B->stride[bnd - 1];
    g.as_layout = o.a_scale_layout; g.bs_layout = o.b_scale_layout;
    if (o.a_scale_layout == MX_SCALE_2D) {
      const int nd = As->ndim;
      g.as_sb = (nd == 3 && batchA > 1) ? As->stride[0] : 0;
      g.as_sm = As->stride[nd - 2]; g.as_sk = As->stride[nd - 1];
    }
    if (o.b_scale_layout == MX_SCALE_2D) {
      const int nd = Bs->ndim;
      g.bs_sb = (nd == 3 && batchB > 1) ? Bs->stride[0] : 0;
      g.bs_sk = Bs->stride[nd - 2]; g.bs_sn = Bs->stride[nd - 1];
    }
    g.c_sb = cnd == 3 ? C->stride[0] : 0; g.c_sm = C->stride[cnd - 2]; g.c_sn = C->stride[cnd - 1];
    return launch_gemm_generic(g, (hipStream_t)stream);
  }

  if (kernel == MX_KERNEL_STREAM) {
    // it uses no workspace, but a caller of MX_KERNEL_AUTO is held to what mx_gemm_workspace_bytes says, whatever is picked
    if (B->dtype != MX_E2M1 && ws_min > 0 && (!workspace || workspace_bytes < ws_min))
      return set_error(MX_ERR_WORKSPACE, "workspace of %lld bytes required, %lld given", (long long)ws_min,
                       (long long)workspace_bytes);
    return launch_gemm_stream(sa, (hipStream_t)stream);
  }

  if (kernel == MX_KERNEL_DECODE) {
    if (M > kDecodeMaxM)
      return set_error(MX_ERR_SHAPE, "the decode kernel handles M <= %lld (got %lld)", (long long)kDecodeMaxM, (long long)M);
    if (o.a_scale_layout != MX_SCALE_2D || o.b_scale_layout != MX_SCALE_2D || Bs->stride[0] != 1 ||
        As->stride[1] != 1)
      return set_error(MX_ERR_LAYOUT, "the decode kernel reads K-contiguous 2-D scales in place");
    if (A->dtype == MX_E2M1 || B->dtype != MX_E2M1)
      return set_error(MX_ERR_DTYPE, "the decode kernel takes 8-bit activations and FP4 weights");
    if (K % 512 != 0 || N % 16 != 0)
      return set_error(MX_ERR_SHAPE, "the decode kernel needs K %% 512 == 0 and N %% 16 == 0");
    DecodeArgs d = {};
    d.X = (const uint8_t*)A->ptr; d.Xs = (const uint8_t*)As->ptr;
    d.W = (const uint8_t*)B->ptr; d.Ws = (const uint8_t*)Bs->ptr; d.C = C->ptr;
    d.M = (int32_t)M; d.N = (int32_t)N; d.K = (int32_t)K;
    d.ldx = a_ld; d.ldxs = As->stride[0]; d.ldw = b_ld; d.ldws = Bs->stride[1]; d.ldc = C->stride[0];
    d.x_fmt = A->dtype; d.w_fmt = B->dtype; d.c_dtype = C->dtype; d.accumulate = o.accumulate;
    const int c_bytes = C->dtype == MX_BF16 ? 2 : 4;
    // slabs of 32 rows of X and C
    auto launch_slabs = [&](const DecodeArgs& full, int out_bytes) {
      for (int64_t m0 = 0; m0 < M; m0 += 32) {
        DecodeArgs s = full;
        s.X = full.X + m0 * full.ldx; s.Xs = full.Xs + m0 * full.ldxs;
        s.C = (uint8_t*)full.C + m0 * full.ldc * out_bytes;
        s.M = (int32_t)(M - m0 < 32 ? M - m0 : 32);
        if (int rc = launch_gemm_decode(s, (hipStream_t)stream)) return rc;
      }
      return (int)MX_OK;
    };
    return launch_slabs(d, c_bytes);
  }

  // ---- MFMA path: bring the scales into the native layout if they are not ----------------------------
  uint8_t* ws = (uint8_t*)workspace;
  const int64_t need = ws_min;
  if (need > 0 && (!ws || workspace_bytes < need))
    return set_error(MX_ERR_WORKSPACE, "workspace of %lld bytes required, %lld given", (long long)need,
                     (long long)workspace_bytes);
  if (need > 0 && ((uintptr_t)ws) % 256 != 0)
    return set_error(MX_ERR_WORKSPACE, "workspace must be 256-byte aligned");
  const uint32_t* as_native = (const uint32_t*)As->ptr;
  const uint32_t* bs_native = (const uint32_t*)Bs->ptr;
  PackArgs pa, pb;
  int S = 1;
  if (kernel == MX_KERNEL_MFMA_128x128 || kernel == MX_KERNEL_MFMA_256x256 || kernel == MX_KERNEL_MFMA_256x256_W4) {
    S = plan_k_splits(M, N, K, o);
    if (S < 0)
      return set_error(MX_ERR_SHAPE, "split_k = %d needs K (%lld) to be a multiple of %d", o.split_k, (long long)K,
                       512 * o.split_k);
  }
  if (S > 1 && plan) return kPlanNotSimple;
  if (kernel == MX_KERNEL_MFMA_128x128 && o.split_k == 0) S = t128_splits(M, N, K, S, A->dtype == MX_E2M1, B->dtype == MX_E2M1);
  if (S > 1 && acc) return kAccNeedsCopy;
  if (kernel == MX_KERNEL_MFMA_128x128) {
    // scales are read where they are if the kernel can (A alone, or A and B), else re-laid first
    T128Args g = {};
    const bool a_can = o.a_scale_layout == MX_SCALE_2D &&
                       t128_plain_scales(As->ptr, As->stride[0], As->stride[1], M, K, A->dtype, B->dtype);
    const bool b_can = o.b_scale_layout == MX_SCALE_2D &&
                       t128_plain_scales(Bs->ptr, Bs->stride[1], Bs->stride[0], N, K, A->dtype, B->dtype);
    g.a_plain = a_can; g.b_plain = a_can && b_can;
    // (in place however the rows lie, where that pays: the re-layout launch costs a small product a third of its time)
    if (!g.b_plain && o.a_scale_layout == MX_SCALE_2D && o.b_scale_layout == MX_SCALE_2D &&
        t128_any_pays(M, N, K, 1, A->dtype == MX_E2M1 && B->dtype == MX_E2M1) &&
        t128_any_scales(As->stride[0], As->stride[1], M, K) && t128_any_scales(Bs->stride[1], Bs->stride[0], N, K))
      g.a_plain = g.b_plain = kT128ScalesAny;
    const bool pack_a = !g.a_plain && !is_native(o.a_scale_layout), pack_b = !g.b_plain && !is_native(o.b_scale_layout);
    if ((!g.a_plain && !pack_a && o.a_scale_layout != MX_SCALE_NATIVE) || (!g.b_plain && !pack_b && o.b_scale_layout != MX_SCALE_NATIVE))
      return set_error(MX_ERR_LAYOUT, "kernel %d reads native-layout scales of kind %d (MX_SCALE_NATIVE for the "
                       "16x16x128-instruction kernels, MX_SCALE_NATIVE32 for pingpong32 / w4p); pass the matching "
                       "layout or the plain 2-D scales", kernel, MX_SCALE_NATIVE);
    g.A = (const uint8_t*)A->ptr; g.B = (const uint8_t*)B->ptr; g.As = (const uint8_t*)As->ptr; g.Bs = (const uint8_t*)Bs->ptr;
    g.C = C->ptr;
    g.lda = a_ld; g.ldb = b_ld; g.ldas = As->stride[0]; g.ldbs = Bs->stride[1]; g.ldc = C->stride[0];
    g.M = (int32_t)M; g.N = (int32_t)N; g.K = (int32_t)K;
    g.a_fmt = A->dtype; g.b_fmt = B->dtype; g.c_dtype = C->dtype; g.accumulate = o.accumulate; g.acc = acc;
    g.batch = 1; g.k_splits = S; g.a_rows = M;
    if (pack_a) {
      if (int rc = make_pack_args(As, o.a_scale_layout, M, K, ws, kPackA, pa)) return rc;
      g.As = ws;
      ws += mx_packed_scale_bytes(M, K);
    }
    if (pack_b) {
      mx_tensor t = *Bs;
      if (o.b_scale_layout == MX_SCALE_2D) {  // [K/32, N] -> view as [N, K/32]
        t.shape[0] = Bs->shape[1]; t.shape[1] = Bs->shape[0];
        t.stride[0] = Bs->stride[1]; t.stride[1] = Bs->stride[0];
      }
      if (int rc = make_pack_args(&t, o.b_scale_layout, N, K, ws, kPackB, pb)) return rc;
      g.Bs = ws;
      ws += mx_packed_scale_bytes(N, K);
    }
    if ((!g.a_plain && ((uintptr_t)g.As) % 16 != 0) || (!g.b_plain && ((uintptr_t)g.Bs) % 16 != 0))
      return set_error(MX_ERR_LAYOUT, "native scale buffers must be 16-byte aligned");
    if (plan) {
      if ((pack_a && o.a_scale_layout != MX_SCALE_2D) || (pack_b && o.b_scale_layout != MX_SCALE_2D) ||
          (g.a_plain && !g.b_plain) || o.accumulate)
        return kPlanNotSimple;
      plan->g = g;
      plan->pack_a = pack_a; plan->pack_b = pack_b;
      if (pack_a) plan->pa = pa;
      if (pack_b) plan->pb = pb;
      return MX_OK;
    }
    if (pack_a || pack_b)   // one launch for both operands
      if (int rc = launch_pack_scales_pair(pack_a ? &pa : nullptr, pack_b ? &pb : nullptr, (hipStream_t)stream)) return rc;
    if (S == 1) return launch_gemm_t128(g, (hipStream_t)stream);
    g.partial = (float*)ws;
    if (int rc = launch_gemm_t128(g, (hipStream_t)stream)) return rc;
    return launch_splitk_reduce(g.partial, S, M, N, C->ptr, C->stride[0], C->dtype, o.accumulate, (hipStream_t)stream);
  }
  if (S > 1) {
    // ---- split-K: the slices are a batch for the scale re-layout and a second grid dimension for the GEMM
    const int64_t Ks = K / S, kbs = Ks / 32;
    if (int rc = make_pack_args(As, MX_SCALE_2D, M, K, ws, kPackA, pa)) return rc;
    pa.K = Ks; pa.batch = S; pa.s_batch = kbs * pa.s_kb;
    const uint32_t* as_p = (const uint32_t*)ws;
    ws += S * mx_packed_scale_bytes(M, Ks);
    mx_tensor t = *Bs;   // [K/32, N] -> view as [N, K/32]
    t.shape[0] = Bs->shape[1]; t.shape[1] = Bs->shape[0];
    t.stride[0] = Bs->stride[1]; t.stride[1] = Bs->stride[0];
    if (int rc = make_pack_args(&t, MX_SCALE_2D, N, K, ws, kPackB, pb)) return rc;
    pb.K = Ks; pb.batch = S; pb.s_batch = kbs * pb.s_kb;
    const uint32_t* bs_p = (const uint32_t*)ws;
    ws += S * mx_packed_scale_bytes(N, Ks);
    float* partial = (float*)ws;
    if (int rc = launch_pack_scales_pair(&pa, &pb, (hipStream_t)stream)) return rc;
    GemmArgs g = {};
    g.A = (const uint8_t*)A->ptr; g.B = (const uint8_t*)B->ptr; g.As = as_p; g.Bs = bs_p; g.C = partial;
    g.lda = a_ld; g.ldb = b_ld; g.ldc = N;
    g.M = (int32_t)M; g.N = (int32_t)N; g.K = (int32_t)Ks;
    g.a_fmt = A->dtype; g.b_fmt = B->dtype; g.c_dtype = MX_F32; g.accumulate = 0;
    g.a_rows = M;
    g.replicas = 1;
    g.k_splits = S;
    g.as_split_stride = mx_packed_scale_bytes(M, Ks) / 4;
    g.bs_split_stride = mx_packed_scale_bytes(N, Ks) / 4;
    g.c_split_stride = M * N;
    if (int rc = launch_gemm_mfma(g, kernel, (hipStream_t)stream)) return rc;
    return launch_splitk_reduce(partial, S, M, N, C->ptr, C->stride[0], C->dtype, o.accumulate, (hipStream_t)stream);
  }
  // (the decode and general kernels returned above: from here on `kernel` is one that reads a native layout)
  const int native = native_layout_of(kernel);
  const bool pack_a = !is_native(o.a_scale_layout), pack_b = !is_native(o.b_scale_layout);
  if ((!pack_a && o.a_scale_layout != native) || (!pack_b && o.b_scale_layout != native))
    return set_error(MX_ERR_LAYOUT, "kernel %d reads native-layout scales of kind %d (MX_SCALE_NATIVE for the "
                     "16x16x128-instruction kernels, MX_SCALE_NATIVE32 for pingpong32 / w4p); pass the matching "
                     "layout or the plain 2-D scales", kernel, native);
  const bool t32 = native == MX_SCALE_NATIVE32;
  if (pack_a) {
    if (int rc = make_pack_args(As, o.a_scale_layout, M, K, ws, t32 ? kPackTile32 : kPackA, pa)) return rc;
    as_native = (const uint32_t*)ws;
    ws += mx_packed_scale_bytes(M, K);
  }
  if (pack_b) {
    mx_tensor t = *Bs;
    if (o.b_scale_layout == MX_SCALE_2D) {  // [K/32, N] -> view as [N, K/32]
      t.shape[0] = Bs->shape[1]; t.shape[1] = Bs->shape[0];
      t.stride[0] = Bs->stride[1]; t.stride[1] = Bs->stride[0];
    }
    if (int rc = make_pack_args(&t, o.b_scale_layout, N, K, ws, t32 ? kPackTile32 : kPackB, pb)) return rc;
    bs_native = (const uint32_t*)ws;
  }
  if (((uintptr_t)as_native) % 16 != 0 || ((uintptr_t)bs_native) % 16 != 0)
    return set_error(MX_ERR_LAYOUT, "native scale buffers must be 16-byte aligned");
  if (pack_a || pack_b)   // one launch for both operands
    if (int rc = launch_pack_scales_pair(pack_a ? &pa : nullptr, pack_b ? &pb : nullptr, (hipStream_t)stream)) return rc;

  GemmArgs g = {};
  g.A = (const uint8_t*)A->ptr; g.B = (const uint8_t*)B->ptr; g.As = as_native; g.Bs = bs_native; g.C = C->ptr;
  g.lda = a_ld; g.ldb = b_ld; g.ldc = C->stride[0];
  g.M = (int32_t)M; g.N = (int32_t)N; g.K = (int32_t)K;
  g.a_fmt = A->dtype; g.b_fmt = B->dtype; g.c_dtype = C->dtype; g.accumulate = o.accumulate;
  g.a_rows = M;
  g.replicas = 1;
  g.tile_rows = tile_rows;
  if (kernel == MX_KERNEL_MFMA_PINGPONG && o.split_k == 0 && workspace && ((uintptr_t)workspace) % 256 == 0) {
    const int64_t tail = pp_tail_bytes(M, N, K, A->dtype == MX_E2M1 && B->dtype == MX_E2M1, true);
    if (tail > 0 && tile_rows == 256 && workspace_bytes >= need + tail) g.tail = (float*)((uint8_t*)workspace + need);
  }
  return launch_gemm_mfma(g, kernel, (hipStream_t)stream);
}
}  // namespace

namespace {
// logical (M, N, K) of a problem from its operand descriptors (FP4 operands count elements, not bytes)
void problem_dims(const mx_tensor& A, const mx_tensor& B, int64_t& M, int64_t& N, int64_t& K) {
  const int an = A.ndim, bn = B.ndim;
  M = an >= 2 ? A.shape[an - 2] : 0;
  K = an >= 2 ? A.shape[an - 1] : 0;
  N = bn >= 2 ? B.shape[bn - 1] : 0;
}
}  // namespace

int64_t mx_static_scratch_bytes(void) { return MX_STATIC_SCRATCH_BYTES; }

int mx_gemm_static(const mx_tensor* A, const mx_tensor* As, const mx_tensor* B, const mx_tensor* Bs, mx_tensor* C,
                   const mx_gemm_opts* opts, void* stream) {
  if (!A || !B) return set_error(MX_ERR_INVALID, "mx_gemm_static: null descriptor");
  if (A->ndim < 2 || A->ndim > 3 || B->ndim < 2 || B->ndim > 3)
    return set_error(MX_ERR_SHAPE, "mx_gemm_static: A and B must have 2 or 3 dimensions");
  int64_t M, N, K;
  problem_dims(*A, *B, M, N, K);
  mx_gemm_opts o = opts_for_room(M, N, K, opts ? *opts : kDefaultOpts, MX_STATIC_SCRATCH_BYTES);
  int64_t need = gemm_workspace_min(M, N, K, o);
  // (here an automatic split gives way to the scales beside it as well)
  if (need > MX_STATIC_SCRATCH_BYTES && o.split_k == 0 && held_partial_sums(M, N, K, o) <= MX_STATIC_SCRATCH_BYTES) {
    o.split_k = 1;
    need = gemm_workspace_min(M, N, K, o);
  }
  if (need > MX_STATIC_SCRATCH_BYTES)
    return set_error(MX_ERR_WORKSPACE, "mx_gemm_static: this problem needs %lld bytes of scratch, the static buffer "
                     "holds %lld; use mx_gemm with a caller-owned workspace", (long long)need,
                     (long long)MX_STATIC_SCRATCH_BYTES);
  void* ws = nullptr;
  if (int rc = static_scratch(&ws)) return rc;
  return mx_gemm(A, As, B, Bs, C, &o, ws, MX_STATIC_SCRATCH_BYTES, stream);
}

int64_t mx_gemm_list_workspace_bytes(int32_t count, const mx_tensor* A, const mx_tensor* B,
                                     const mx_gemm_opts* opts) {
  if (count <= 0 || !A || !B) return 0;
  int64_t need = 0;   // every problem has its own slice: the problems of a list run side by side
  for (int32_t i = 0; i < count; ++i) {
    int64_t M, N, K;
    problem_dims(A[i], B[i], M, N, K);
    need += round256(gemm_workspace_min(M, N, K, opts ? *opts : kDefaultOpts));
  }
  return need;
}

int mx_gemm_list(int32_t count, const mx_tensor* A, const mx_tensor* As, const mx_tensor* B, const mx_tensor* Bs,
                 mx_tensor* C, const mx_gemm_opts* opts, void* workspace, int64_t workspace_bytes, void* stream) {
  if (count < 0) return set_error(MX_ERR_INVALID, "mx_gemm_list: negative count");
  if (count == 0) return MX_OK;
  if (!A || !As || !B || !Bs || !C) return set_error(MX_ERR_INVALID, "mx_gemm_list: null descriptor array");
  std::vector<int64_t> share(count);   // of the workspace
  int64_t need = 0;
  auto shares = [&](int64_t (*bytes)(int64_t, int64_t, int64_t, const mx_gemm_opts&)) {
    need = 0;
    for (int32_t i = 0; i < count; ++i) {
      int64_t M, N, K;
      problem_dims(A[i], B[i], M, N, K);
      need += share[i] = round256(bytes(M, N, K, opts ? *opts : kDefaultOpts));
    }
  };
  shares(gemm_workspace_min);
  if ((workspace ? workspace_bytes : 0) < need) shares(gemm_workspace_held);
  if (need > 0 && (!workspace || workspace_bytes < need))
    return set_error(MX_ERR_WORKSPACE, "workspace of %lld bytes required, %lld given", (long long)need,
                     (long long)workspace_bytes);
  if (need > 0 && ((uintptr_t)workspace) % 256 != 0) return set_error(MX_ERR_WORKSPACE, "workspace must be 256-byte aligned");

  // Pass 1: validate everything and sort the problems: those that would run on the 128 x 128 one-tile kernel are
  // collected (no launch), the others are remembered for a call of their own.  Nothing is enqueued if any problem
  // is invalid.
  struct Item { int32_t index; int64_t ws_off, ws_bytes; bool simple; GemmPlan plan; };
  std::vector<Item> items;
  items.reserve(count);
  int64_t off = 0;
  for (int32_t i = 0; i < count; ++i) {
    int64_t M, N, K;
    problem_dims(A[i], B[i], M, N, K);
    const int64_t b = share[i];
    Item it = {};
    it.index = i; it.ws_off = off; it.ws_bytes = b;
    off += b;
    if (A[i].ndim == 2 && B[i].ndim == 2 && (M == 0 || N == 0)) continue;   // empty problem
    const int rc = gemm_impl(&A[i], &As[i], &B[i], &Bs[i], &C[i], opts, (uint8_t*)workspace + it.ws_off, it.ws_bytes,
                             stream, &it.plan);
    if (rc < 0) {
      char inner[400];
      snprintf(inner, sizeof inner, "%s", mx_last_error());
      return set_error(rc, "problem %d of the list: %s", (int)i, inner);
    }
    it.simple = rc == MX_OK;
    items.push_back(it);
  }
  // Pass 2: one scale re-layout launch per 64 scale tensors, one persistent GEMM launch per 32 problems of one
  // element-format pair
  std::vector<PackArgs> packs;
  for (const Item& it : items) {
    if (!it.simple) continue;
    if (it.plan.pack_a) packs.push_back(it.plan.pa);
    if (it.plan.pack_b) packs.push_back(it.plan.pb);
  }
  if (!packs.empty())
    if (int rc = launch_pack_scales_list(packs.data(), (int)packs.size(), (hipStream_t)stream)) return rc;
  std::vector<char> done(items.size(), 0);
  for (size_t i = 0; i < items.size(); ++i) {
    if (!items[i].simple || done[i]) continue;
    std::vector<T128Args> group;
    const T128Args& g0 = items[i].plan.g;
    for (size_t j = i; j < items.size(); ++j) {
      const T128Args& g = items[j].plan.g;
      if (items[j].simple && !done[j] && g.a_fmt == g0.a_fmt && g.b_fmt == g0.b_fmt) {
        group.push_back(g);
        done[j] = 1;
      }
    }
    // longest products first: a workgroup's second tile is then a short one
    std::stable_sort(group.begin(), group.end(), [](const T128Args& x, const T128Args& y) { return x.K > y.K; });
    if (int rc = launch_gemm_t128_list(group.data(), (int)group.size(), (hipStream_t)stream)) return rc;
  }
  // Pass 3: the rest (large problems for the persistent 256 x 256 kernel, skinny ones for the decode kernel,
  // split-K, batched operands, layouts only the general kernel reads), one call each
  for (const Item& it : items) {
    if (it.simple) continue;
    const int32_t i = it.index;
    const int rc = mx_gemm(&A[i], &As[i], &B[i], &Bs[i], &C[i], opts, (uint8_t*)workspace + it.ws_off, it.ws_bytes, stream);
    if (rc != MX_OK) {
      char inner[400];
      snprintf(inner, sizeof inner, "%s", mx_last_error());
      return set_error(rc, "problem %d of the list: %s", (int)i, inner);
    }
  }
  return MX_OK;
}

int mx_bench_gemm(int32_t nsets, const mx_tensor* A, const mx_tensor* As, const mx_tensor* B, const mx_tensor* Bs,
                  mx_tensor* C, const mx_gemm_opts* opts, void* workspace, int64_t workspace_bytes, int32_t warmup,
                  int32_t iters, float* times_ms, void* stream) {
  if (nsets <= 0 || !A || !As || !B || !Bs || !C) return set_error(MX_ERR_INVALID, "mx_bench_gemm: no operand sets");
  if (warmup < 0 || iters <= 0 || iters > 65536 || !times_ms)
    return set_error(MX_ERR_INVALID, "mx_bench_gemm: iters must be in 1..65536 and times_ms non-null");
  hipStream_t st = (hipStream_t)stream;
  for (int i = 0; i < warmup; ++i) {
    const int s = i % nsets;
    if (int rc = mx_gemm(&A[s], &As[s], &B[s], &Bs[s], &C[s], opts, workspace, workspace_bytes, stream)) return rc;
  }
  hipEvent_t* ev = (hipEvent_t*)calloc((size_t)2 * iters, sizeof(hipEvent_t));
  if (!ev) return set_error(MX_ERR_INVALID, "mx_bench_gemm: out of host memory");
  int rc = MX_OK, made = 0;
  for (; made < 2 * iters; ++made)
    if (hipEventCreate(&ev[made]) != hipSuccess) { rc = set_error(MX_ERR_DEVICE, "mx_bench_gemm: hipEventCreate failed"); break; }
  for (int i = 0; rc == MX_OK && i < iters; ++i) {
    const int s = (warmup + i) % nsets;
    if (hipEventRecord(ev[2 * i], st) != hipSuccess) { rc = set_error(MX_ERR_DEVICE, "mx_bench_gemm: hipEventRecord failed"); break; }
    rc = mx_gemm(&A[s], &As[s], &B[s], &Bs[s], &C[s], opts, workspace, workspace_bytes, stream);
    if (rc == MX_OK && hipEventRecord(ev[2 * i + 1], st) != hipSuccess)
      rc = set_error(MX_ERR_DEVICE, "mx_bench_gemm: hipEventRecord failed");
  }
  // the stream is drained on every path, so that no event is destroyed while still pending
  const hipError_t es = hipStreamSynchronize(st);
  if (rc == MX_OK && es != hipSuccess) rc = set_error(MX_ERR_DEVICE, "mx_bench_gemm: %s", hipGetErrorString(es));
  for (int i = 0; rc == MX_OK && i < iters; ++i)
    if (hipEventElapsedTime(&times_ms[i], ev[2 * i], ev[2 * i + 1]) != hipSuccess)
      rc = set_error(MX_ERR_DEVICE, "mx_bench_gemm: hipEventElapsedTime failed");
  for (int i = 0; i < made; ++i) (void)hipEventDestroy(ev[i]);
  free(ev);
  return rc;
}

namespace {
// slots_in_use: on the device, may be null (all num_slots); slots beyond it hold no routed row
int gemm_grouped_impl(const mx_tensor* A, const mx_tensor* As, const mx_tensor* W, const mx_tensor* Ws,
                      mx_tensor* C, const float* topk_weights, const int32_t* sorted_token_ids,
                      int64_t num_slots, const int32_t* slots_in_use, const int32_t* sorted_expert_ids, int32_t tile_m,
                      int32_t num_token_replicas, int64_t num_valid_ids, const mx_gemm_opts* opts,
                      void* workspace, int64_t workspace_bytes, void* stream) {
  const mx_gemm_opts& o = opts ? *opts : kDefaultOpts;
  if (int rc = check_tensor(A, "A", 2, 2)) return rc;
  if (int rc = check_tensor(As, "A_scale", 2, 2)) return rc;
  if (int rc = check_tensor(W, "W", 3, 3)) return rc;
  if (int rc = check_tensor(Ws, "W_scale", 3, 3)) return rc;
  if (int rc = check_tensor(C, "C", 2, 2)) return rc;
  if (!sorted_token_ids || !sorted_expert_ids) return set_error(MX_ERR_INVALID, "null index arrays");
  if (tile_m <= 0 || num_slots % tile_m != 0)
    return set_error(MX_ERR_SHAPE, "num_slots (%lld) must be a multiple of tile_m (%d)", (long long)num_slots, tile_m);
  if (num_token_replicas <= 0) return set_error(MX_ERR_INVALID, "num_token_replicas must be positive");
  if (!is_elem(A->dtype) || !is_elem(W->dtype)) return set_error(MX_ERR_DTYPE, "A/W must be MX element formats");
  if (As->dtype != MX_E8M0 || Ws->dtype != MX_E8M0) return set_error(MX_ERR_DTYPE, "scales must be MX_E8M0");
  if (C->dtype != MX_F32 && C->dtype != MX_BF16) return set_error(MX_ERR_DTYPE, "C must be MX_F32 or MX_BF16");
  if (o.block_size != 32) return set_error(MX_ERR_INVALID, "grouped GEMM supports block size 32 only");
  const int64_t T = A->shape[0], K = A->shape[1], E = W->shape[0], N = W->shape[1];
  if (W->shape[2] != K)
    return set_error(MX_ERR_SHAPE, "Incompatible matrices: K dimension of A (%lld) must match K dimension of W (%lld)",
                     (long long)K, (long long)W->shape[2]);
  if (K % 32 != 0) return set_error(MX_ERR_SHAPE, "K (%lld) must be a multiple of 32", (long long)K);
  const int64_t KB = K / 32;
  if (As->shape[0] != T || As->shape[1] != KB) return set_error(MX_ERR_SHAPE, "A_scale must be [tokens, K/32]");
  if (!is_native(o.b_scale_layout) && (Ws->shape[0] != E || Ws->shape[1] != N || Ws->shape[2] != KB))
    return set_error(MX_ERR_SHAPE, "W_scale must be [experts, N, K/32]");
  if (C->shape[1] != N || C->shape[0] < num_valid_ids)
    return set_error(MX_ERR_SHAPE, "C must be [>= num_valid_ids, N]");
  if ((num_valid_ids + num_token_replicas - 1) / num_token_replicas > T)
    return set_error(MX_ERR_SHAPE, "num_valid_ids / num_token_replicas exceeds the rows of A");
  if (num_slots == 0 || N == 0) return MX_OK;
  if (E <= 0 || E > 0x7FFFFFFF) return set_error(MX_ERR_SHAPE, "W must hold at least one expert");
  if (A->dtype == MX_E2M1 && A->packed_dim != 1) return set_error(MX_ERR_LAYOUT, "A must be packed along K");
  if (W->dtype == MX_E2M1 && W->packed_dim != 2) return set_error(MX_ERR_LAYOUT, "W must be packed along K");

  const char* why = nullptr;
  if (!pair_supported_by_mfma(A->dtype, W->dtype)) why = "element format pair not instantiated";
  else if ((why = mfma_operand_issue(A->ptr, T, K, A->stride[0], A->stride[1], A->dtype, 1))) {}
  else if ((why = mfma_operand_issue(W->ptr, N, K, W->stride[1], W->stride[2], W->dtype, 1))) {}
  else if (W->stride[0] % 16 != 0) why = "expert pitch of W is not a multiple of 16 bytes";
  else if (C->stride[1] != 1) why = "C is not row-major";
  else if (tile_m % 128 != 0) why = "tile_m is not a multiple of 128";
  else if (o.a_scale_layout != MX_SCALE_2D) why = "A_scale must be the plain 2-D layout";

  int kernel = o.kernel;
  if (kernel == MX_KERNEL_AUTO) {
    if (why) kernel = MX_KERNEL_GENERIC;
    else kernel = (tile_m % 256 == 0 && N > 128) ? big_tile_kernel() : MX_KERNEL_MFMA_128x128;
  } else if (kernel != MX_KERNEL_GENERIC) {
    if (why) return set_error(MX_ERR_LAYOUT, "requested kernel %d cannot run this problem: %s", kernel, why);
    const int bm = kernel == MX_KERNEL_MFMA_128x128 ? 128 : 256;
    if (kernel == MX_KERNEL_DECODE || tile_m % bm != 0)
      return set_error(MX_ERR_LAYOUT, "kernel %d needs tile_m to be a multiple of its row tile", kernel);
  }

  if (kernel == MX_KERNEL_GENERIC) {
    if (o.a_scale_layout != MX_SCALE_2D || o.b_scale_layout != MX_SCALE_2D)
      return set_error(MX_ERR_LAYOUT, "the generic grouped kernel reads plain 2-D / 3-D scales");
    GenericArgs g = {};
    g.A = (const uint8_t*)A->ptr; g.As = (const uint8_t*)As->ptr;
    g.B = (const uint8_t*)W->ptr; g.Bs = (const uint8_t*)Ws->ptr; g.C = C->ptr;
    g.batch = 1; g.M = (int32_t)T; g.N = (int32_t)N; g.K = (int32_t)K; g.block = 32;
    g.a_fmt = A->dtype; g.b_fmt = W->dtype; g.scale_fmt = MX_E8M0; g.c_dtype = C->dtype; g.accumulate = o.accumulate;
    g.a_packed_k = 1; g.b_packed_k = 1;
    g.a_sm = A->stride[0]; g.a_sk = A->stride[1];
    g.as_sm = As->stride[0]; g.as_sk = As->stride[1];
    g.b_sn = W->stride[1]; g.b_sk = W->stride[2]; g.b_se = W->stride[0];
    g.bs_sn = Ws->stride[1]; g.bs_sk = Ws->stride[2]; g.bs_se = Ws->stride[0];
    g.c_sm = C->stride[0]; g.c_sn = C->stride[1];
    g.sorted_token_ids = sorted_token_ids; g.sorted_expert_ids = sorted_expert_ids; g.topk_weights = topk_weights;
    g.tile_m = tile_m; g.replicas = num_token_replicas; g.num_valid_ids = num_valid_ids; g.num_slots = num_slots;
    g.num_experts = (int32_t)E;
    return launch_gemm_generic(g, (hipStream_t)stream);
  }

  uint8_t* ws = (uint8_t*)workspace;
  const int64_t need = grouped_workspace_min(num_slots, N, K, E, o);
  if (!ws || workspace_bytes < need)
    return set_error(MX_ERR_WORKSPACE, "workspace of %lld bytes required, %lld given", (long long)need,
                     (long long)workspace_bytes);
  if (((uintptr_t)ws) % 256 != 0) return set_error(MX_ERR_WORKSPACE, "workspace must be 256-byte aligned");
  if (kernel == MX_KERNEL_MFMA_128x128) {
    T128Args g = {};
    g.a_plain = t128_plain_scales(As->ptr, As->stride[0], As->stride[1], T, K, A->dtype, W->dtype);
    PackArgs pa = {}, pw;
    g.As = (const uint8_t*)As->ptr; g.ldas = As->stride[0];
    if (!g.a_plain) {   // gathered into slot order while re-laying
      pa.target = kPackA;
      pa.src = (const uint8_t*)As->ptr; pa.dst = (uint32_t*)ws;
      pa.rows = num_slots; pa.K = K; pa.s_row = As->stride[0]; pa.s_kb = As->stride[1];
      pa.layout = MX_SCALE_2D; pa.batch = 1;
      pa.gather_ids = sorted_token_ids; pa.replicas = num_token_replicas; pa.num_valid_ids = num_valid_ids;
      g.As = ws;
      ws += mx_packed_scale_bytes(num_slots, K);
    }
    g.Bs = (const uint8_t*)Ws->ptr;
    const bool pack_w = !is_native(o.b_scale_layout);
    if (!pack_w && o.b_scale_layout != MX_SCALE_NATIVE)
      return set_error(MX_ERR_LAYOUT, "kernel %d reads native-layout scales of kind %d, W_scale has kind %d", kernel,
                       MX_SCALE_NATIVE, o.b_scale_layout);
    if (E * mx_packed_scale_bytes(N, K) >= ((int64_t)1 << 31))
      return set_error(MX_ERR_SHAPE, "the packed scales of all experts must stay below 2 GiB");
    if (pack_w) {
      if (o.b_scale_layout != MX_SCALE_2D) return set_error(MX_ERR_LAYOUT, "W_scale must be [E, N, K/32] or native");
      if (int rc = make_pack_args(Ws, MX_SCALE_2D, N, K, ws, kPackB, pw)) return rc;
      g.Bs = ws;
    }
    if (T == 0) return MX_OK;   // no slot holds a row (the descriptor of A ends behind the last one: there has to be one)
    if (!g.a_plain || pack_w)
      if (int rc = launch_pack_scales_pair(g.a_plain ? nullptr : &pa, pack_w ? &pw : nullptr, (hipStream_t)stream)) return rc;
    g.A = (const uint8_t*)A->ptr; g.B = (const uint8_t*)W->ptr; g.C = C->ptr;
    g.lda = A->stride[0]; g.ldb = W->stride[1]; g.ldc = C->stride[0];
    g.M = (int32_t)num_slots; g.N = (int32_t)N; g.K = (int32_t)K;
    g.a_fmt = A->dtype; g.b_fmt = W->dtype; g.c_dtype = C->dtype; g.accumulate = o.accumulate;
    g.batch = 1; g.k_splits = 1;
    g.sorted_token_ids = sorted_token_ids; g.sorted_expert_ids = sorted_expert_ids; g.topk_weights = topk_weights;
    g.tile_m = tile_m; g.replicas = num_token_replicas; g.num_valid_ids = num_valid_ids; g.num_experts = (int32_t)E;
    g.a_rows = T; g.b_expert = W->stride[0]; g.bs_expert = mx_packed_scale_bytes(N, K);
    return launch_gemm_t128(g, (hipStream_t)stream);
  }
  // A scales: gathered into slot order while re-laying; W scales of all experts ride in the same launch
  const int native = native_layout_of(kernel);
  const bool t32 = native == MX_SCALE_NATIVE32;
  PackArgs pa = {}, pw;
  pa.target = t32 ? kPackTile32 : kPackA;
  pa.src = (const uint8_t*)As->ptr; pa.dst = (uint32_t*)ws;
  pa.rows = num_slots; pa.K = K; pa.s_row = As->stride[0]; pa.s_kb = As->stride[1];
  pa.layout = MX_SCALE_2D; pa.batch = 1;
  pa.gather_ids = sorted_token_ids; pa.replicas = num_token_replicas; pa.num_valid_ids = num_valid_ids;
  const uint32_t* as_native = (const uint32_t*)ws;
  ws += mx_packed_scale_bytes(num_slots, K);
  const uint32_t* bs_native = (const uint32_t*)Ws->ptr;
  const bool pack_w = !is_native(o.b_scale_layout);
  if (!pack_w && o.b_scale_layout != native)
    return set_error(MX_ERR_LAYOUT, "kernel %d reads native-layout scales of kind %d, W_scale has kind %d", kernel,
                     native, o.b_scale_layout);
  if (E * mx_packed_scale_bytes(N, K) >= ((int64_t)1 << 31))
    return set_error(MX_ERR_SHAPE, "the packed scales of all experts must stay below 2 GiB");
  if (pack_w) {
    if (o.b_scale_layout != MX_SCALE_2D) return set_error(MX_ERR_LAYOUT, "W_scale must be [E, N, K/32] or native");
    if (int rc = make_pack_args(Ws, MX_SCALE_2D, N, K, ws, t32 ? kPackTile32 : kPackB, pw)) return rc;
    bs_native = (const uint32_t*)ws;
  }
  if (T == 0) return MX_OK;   // (as above)
  if (int rc = launch_pack_scales_pair(&pa, pack_w ? &pw : nullptr, (hipStream_t)stream)) return rc;
  GemmArgs g = {};
  g.A = (const uint8_t*)A->ptr; g.B = (const uint8_t*)W->ptr; g.As = as_native; g.Bs = bs_native; g.C = C->ptr;
  g.lda = A->stride[0]; g.ldb = W->stride[1]; g.ldc = C->stride[0];
  g.M = (int32_t)num_slots; g.N = (int32_t)N; g.K = (int32_t)K;
  g.a_fmt = A->dtype; g.b_fmt = W->dtype; g.c_dtype = C->dtype; g.accumulate = o.accumulate;
  g.sorted_token_ids = sorted_token_ids; g.sorted_expert_ids = sorted_expert_ids; g.topk_weights = topk_weights;
  g.tile_m = tile_m; g.replicas = num_token_replicas; g.num_valid_ids = num_valid_ids;
  g.num_experts = (int32_t)E;
  g.b_expert_stride = W->stride[0];
  g.bs_expert_stride = mx_packed_scale_bytes(N, K) / 4;
  g.a_rows = T;
  g.num_slots = slots_in_use;
  if (kernel == MX_KERNEL_MFMA_PINGPONG) {
    const int64_t tail = pp_tail_bytes(num_slots, N, K, A->dtype == MX_E2M1 && W->dtype == MX_E2M1, !slots_in_use);
    if (tail > 0 && workspace_bytes >= need + tail) g.tail = (float*)((uint8_t*)workspace + need);
  }
  return launch_gemm_mfma(g, kernel, (hipStream_t)stream);
}
}  // namespace

int mx_gemm_grouped(const mx_tensor* A, const mx_tensor* As, const mx_tensor* W, const mx_tensor* Ws,
                    mx_tensor* C, const float* topk_weights, const int32_t* sorted_token_ids,
                    int64_t num_slots, const int32_t* sorted_expert_ids, int32_t tile_m,
                    int32_t num_token_replicas, int64_t num_valid_ids, const mx_gemm_opts* opts,
                    void* workspace, int64_t workspace_bytes, void* stream) {
  return gemm_grouped_impl(A, As, W, Ws, C, topk_weights, sorted_token_ids, num_slots, nullptr, sorted_expert_ids, tile_m,
                           num_token_replicas, num_valid_ids, opts, workspace, workspace_bytes, stream);
}

int64_t mx_moe_align_max_slots(int64_t num_ids, int32_t num_experts, int32_t tile_m) {
  if (num_ids < 0 || num_experts <= 0 || tile_m <= 0) return 0;
  const int64_t nonempty = num_experts < num_ids ? num_experts : num_ids;
  return (num_ids + nonempty * (tile_m - 1)) / tile_m * tile_m;
}

int64_t mx_moe_align_workspace_bytes(int64_t num_ids, int32_t num_experts) {
  if (num_ids <= 0 || num_experts <= 0) return 0;
  return round256(moe_align_workspace_bytes(num_ids, num_experts));
}

int mx_moe_align(const int32_t* topk_ids, int64_t num_ids, int32_t num_experts, int32_t tile_m,
                 int32_t* sorted_token_ids, int32_t* sorted_expert_ids, int32_t* num_slots_out, void* workspace,
                 int64_t workspace_bytes, void* stream) {
  if (num_ids < 0 || num_experts <= 0 || tile_m <= 0) return set_error(MX_ERR_INVALID, "moe_align: bad sizes");
  if (num_ids >= 0x7FFFFFFF) return set_error(MX_ERR_SHAPE, "moe_align: too many ids");
  const int64_t max_slots = mx_moe_align_max_slots(num_ids, num_experts, tile_m);
  if (max_slots == 0) {
    return MX_OK;
  }
  if (max_slots >= 0x7FFFFFFF) return set_error(MX_ERR_SHAPE, "moe_align: too many slots");
  if (!topk_ids || !sorted_token_ids || !sorted_expert_ids) return set_error(MX_ERR_INVALID, "moe_align: null pointer");
  const int64_t need = moe_align_workspace_bytes(num_ids, num_experts);
  if (need > 0 && (!workspace || workspace_bytes < need))
    return set_error(MX_ERR_WORKSPACE, "moe_align: workspace of %lld bytes required, %lld given", (long long)need,
                     (long long)workspace_bytes);
  if (need > 0 && ((uintptr_t)workspace) % 4 != 0) return set_error(MX_ERR_WORKSPACE, "moe_align: workspace must be 4-byte aligned");
  return launch_moe_align(topk_ids, 0, num_ids, num_experts, tile_m, sorted_token_ids, sorted_expert_ids,
                          num_slots_out, max_slots, (int32_t*)workspace, (hipStream_t)stream);
}

namespace {
// Sizes of a mixture-of-experts layer and where its pieces lie in the workspace.
struct MoePlan {
  int64_t T, n, E, H, F, H_out;
  bool stream;          // experts' weights streamed for a few rows each
  bool tiles;           // row tiles of their own (mx_moe_tile.hip); neither: grouped GEMMs on aligned slots
  int32_t splits;       // tiles: K ranges of the down projection
  int64_t max_tiles, info;
  int32_t tile_m;
  int64_t q, qs, c3, c1, slots, in_use, max_slots, blocks, align, grouped, grouped_bytes, total;   // offsets (bytes)
};
// Rows per expert up to which the weights are streamed where the row tiles below do not take the layer.  us per layer, streamed | grouped with 256-slot tiles:
//   16 experts of 4096 x 4096, FP8: 32 rows 218 | 266, 64 rows 336 | 283; FP4: 32 rows 139 | 183, 48 rows 173 | 187, 64 rows
//   238 | 193
//   8 experts of 4096 x 14336, FP8: 16 rows 231 | 358, 32 rows 372 | 366; FP4: 32 rows 239 | 282, 48 rows 274 | 286
//   64 experts of 3584 x 1024, FP8: 32 rows 223 | 248
// (128-slot and 64-slot tiles are slower than one or the other everywhere.)  Beyond 32 rows an expert's weights are read once
// more; against that stand the tiles' extra passes, some 40 us whatever the size.  33, 40 and 48 rows:
//   0.81 GB: 8 experts 226 | 282, 245 | 284, 262 | 286; 16 experts 234 | 254, 252 | 257, 269 | 261
//   0.96 GB: 8 experts 260 | 303, 310 | 305, 315 | 310
//   1.06 GB: 8 experts 294 | 307, 311 | 309, 389 | 314;  1.11 GB: 16 experts 289 | 286, 358 | 290, 374 | 294, 32 experts 294 |
//     314, 368 | 320, 384 | 325
//   1.21 GB: 8 experts 289 | 318 (34 rows 336 | 321), 360 | 321, 392 | 327;  1.41 GB: 8 experts 357 | 360 (34 rows 384 | 362), 416 | 365,
//     455 | 369; FP4, 16 experts 421 | 430, 505 | 437, 516 | 442
// so that the tiles are ahead from 1 GB of weights on, at 33 rows not yet everywhere.
// (64 rows: with a longer list of ids, mx_stream.h.)
constexpr int64_t kMoeStreamRows = 48, kMoeStreamTwiceBytes = 1000000000;

// what keeps a layer from the row tiles of mx_moe_tile.hip (nullptr: nothing): both weights' scales packed, whole K-steps and
// column tiles, a routing that one workgroup sorts out, and no padding asked for, which they don't have
const char* moe_tiles_issue(const MoePlan& p, const mx_gemm_opts& o) {
  if (o.a_scale_layout != MX_SCALE_NATIVE || o.b_scale_layout != MX_SCALE_NATIVE) return "scales are not packed";
  if (p.H % 128 != 0 || p.F % 128 != 0) return "H or F is not a multiple of 128";
  if (p.n > kMoeTileMaxIds || p.E > kMoeTileMaxExperts) return "too many ids or experts";
  if (o.tile_m != 0) return "tile_m";
  return nullptr;
}

// Rows per expert on average up to which the row tiles are mostly not behind the 256-row tiles, which need more launches around them.  Random routing
// gives some experts one tile of 64 (FP4 and long rows 128) more than the average; where the layer is large that is at once another round of
// workgroups, while 256-row tiles still have one each.  us, row tiles | 256-row tiles, random routing, at the rows in front:
//   long rows, FP8 beyond 1 GB of weights.  96: 8 experts of 4096 x 14336 381 | 384 (at 112 and 128 no longer), 16 of 3072 x 8192 349 | 350, 64 of 3072 x
//     2048 377 | 384, 16 of 4096 x 7168 392 | 373.  Larger ones, 64, 72 and 88: 16 of 4096 x 8192 392 | 400, 422 | 405, 438 | 414; 12 of 3584 x 14336 440 |
//     473, 515 | 478, 512 | 488; 32 of 3584 x 8192 658 | 642, 714 | 653, 769 | 671; 32 of 4096 x 4096 (1.6 GB) 404 | 426, 432 | 432, 447 | 448
//   long rows, many experts.  120 and 128: 16 of 2560 x 4096 FP8 202 | 194, 210 | 197; 16 of 4096 x 4096 FP8 268 | 289, 287 | 292, FP4 183 | 190, 212 | 198; 16 of
//     3584 x 8192 FP4 293 | 302, 370 | 306; 32 of 4096 x 4096 FP4 353 | 346, 391 | 353.  Others: 8 of 4096 x 7168 FP8 241 | 255, 244 | 259, FP4 160 |
//     191, 187 | 194; 8 of 4096 x 14336 FP4 294 | 317, 322 | 320; 32 of 4096 x 2048 FP8 278 | 303, 292 | 307, FP4 201 | 214, 222 | 218
//   short rows, large layers.  72 and 88: 32 of 1536 x 8192 FP8 398 | 367, 397 | 378, FP4 297 | 289, 312 | 299; 32 of 2048 x 8192 FP8 452 | 441, 478 | 455; 64 of
//     2048 x 4096 FP8 456 | 469, 470 | 484, FP4 345 | 353, 363 | 367; 64 of 1024 x 4096, 88 and 112: FP8 309 | 305, 320 | 321, FP4 249 | 242, 268 | 256.
//     Medium ones of many experts, 120 and 128: 32 of 1536 x 4096 FP8 246 | 235, 265 | 239, FP4 198 | 191, 214 | 194; 128 of 1536 x 1024 FP8 295 | 288, 311 |
//     292; 64 of 2048 x 2048 FP8 290 | 298, 306 | 303
//   short rows, small layers, a third tile of 64.  136 and 160: 8 of 1024 x 7168 FP8 112 | 129, 115 | 125, FP4 87 | 112, 91 | 114; 32 of 1024 x 2048 FP8 (144) 120 |
//     126, 123 | 129; 16 of 1024 x 8192 FP8 203 | 200, 215 | 209, FP4 165 | 173, 174 | 184; 8 of 2048 x 8192 FP8 172 | 182, 178 | 186; 16 of 2048 x 4096 FP8
//     166 | 174, 176 | 181; 64 of 2048 x 1024 FP8 197 | 205, 212 | 217.  Not: 32 of 1024 x 4096 FP8 203 | 197, 213 | 205; 64 of 1024 x 2048 FP8 208 |
//     200, 227 | 212; 8 of 2048 x 14336 FP8 283 | 261, 295 | 269, FP4 223 | 215, 232 | 224; 16 of 1280 x 8192 FP8 249 | 239, 267 | 248; 32 of 1536 x 2048
//     FP4 132 | 125, 141 | 131; 32 of 2048 x 2048 FP4 146 | 138, 156 | 145; 64 of 1536 x 1024 FP4 154 | 148, 168 | 156 (12 columns for eight XCDs)
// Where one expert has half of the copies or the popularity falls with the rank the row tiles are further ahead: 8 of 4096 x 14336 FP4, 96 rows
// on average 278 | 328, 290 | 335.
int64_t moe_tile_limit(const MoePlan& p, int64_t weight_bytes, bool fp4) {
  const int64_t cols = p.E * p.F;
  if (p.H > 2048) {
    if (!fp4 && weight_bytes > kMoeStreamTwiceBytes) return weight_bytes > 1500000000 ? 64 : 96;
    return p.E >= 16 && (p.F >= 4096 || cols > 65536) ? 120 : 128;
  }
  if (cols > 196608) return p.H <= 1024 ? 96 : 72;
  if (p.H <= 1024 && cols <= 131072 && (p.E <= 16 || cols < 131072)) return 160;
  if (cols <= 65536 && (p.E <= 16 || (p.F <= 1024 && p.H_out % 1024 == 0))) return 160;
  return p.H > 1024 && p.E >= 32 && cols >= 131072 ? 120 : 128;
}

MoePlan moe_plan(int64_t T, int32_t topk, const mx_tensor& W1, const mx_tensor& W2, const mx_gemm_opts& o, int32_t max_splits = 8) {
  MoePlan p = {};
  p.T = T; p.n = T * topk; p.E = W1.shape[0]; p.H = W1.shape[2]; p.F = W1.shape[1] / 2; p.H_out = W2.shape[1];
  const int64_t weights = p.E * (2 * p.F * p.H + p.H_out * p.F) / (W1.dtype == MX_E2M1 ? 2 : 1);   // bytes
  const int64_t rows = weights > kMoeStreamTwiceBytes ? 32 : kMoeStreamRows;
  p.stream = p.n <= kMoeMaxIds && p.n <= p.E * rows && p.H % 128 == 0 && p.F % 128 == 0;
  // Row tiles where the weights would be streamed more than once and the 256-row tiles are not ahead.
  const bool can_tile = moe_tiles_issue(p, o) == nullptr && p.n <= p.E * moe_tile_limit(p, weights, W1.dtype == MX_E2M1);
  if (can_tile && moe_leaves_streaming(p.n, p.E, topk)) p.stream = false;
  p.tiles = can_tile && !p.stream;
  int64_t off = 0;
  auto take = [&](int64_t bytes) { const int64_t at = off; off += round256(bytes); return at; };
  p.q = take(p.n * p.F);
  p.qs = take(p.n * (p.F / 32));
  if (p.tiles) p.tile_m = moe_tile_rows(p.n, p.E, p.H, W1.dtype);
  p.splits = p.tiles ? moe_tile_splits(p.n, p.E, p.tile_m, p.H_out, p.F) : 1;
  if (p.splits > max_splits) p.splits = max_splits;
  p.c3 = take(p.n * p.H_out * 4 * p.splits);
  if (p.tiles) {
    p.max_tiles = moe_tiles_max(p.n, p.E, p.tile_m);
    p.info = take(p.max_tiles * (int64_t)sizeof(MoeTile));
    p.slots = take(p.max_tiles * p.tile_m * 4);
  } else if (!p.stream) {
    p.tile_m = o.tile_m > 0 ? o.tile_m : 256;
    p.max_slots = mx_moe_align_max_slots(p.n, (int32_t)p.E, p.tile_m);
    p.c1 = take(p.n * p.F * 4);
    p.slots = take(p.max_slots * 4);
    p.in_use = take(4);
    p.blocks = take(p.max_slots / p.tile_m * 4);
    p.align = take(mx_moe_align_workspace_bytes(p.n, (int32_t)p.E));
    mx_gemm_opts g1 = kDefaultOpts, g2 = kDefaultOpts;
    g1.b_scale_layout = o.a_scale_layout;
    g2.b_scale_layout = o.b_scale_layout;
    const int64_t b1 = mx_gemm_grouped_workspace_bytes(p.max_slots, 2 * p.F, p.H, p.E, &g1);
    const int64_t b2 = mx_gemm_grouped_workspace_bytes(p.max_slots, p.H_out, p.F, p.E, &g2);
    p.grouped_bytes = b1 > b2 ? b1 : b2;
    p.grouped = take(p.grouped_bytes);
  }
  p.total = off;
  return p;
}

inline mx_tensor tensor2d(void* ptr, int dtype, int64_t rows, int64_t cols, int64_t ld) {
  return mx_tensor{ptr, dtype, 2, {rows, cols, 0, 0}, {ld, 1, 0, 0}, -1, 0};
}
}  // namespace

int64_t mx_moe_forward_workspace_bytes(int64_t T, int32_t topk, const mx_tensor* W1, const mx_tensor* W2,
                                       const mx_gemm_opts* opts) {
  if (T <= 0 || topk <= 0 || !W1 || !W2 || W1->ndim != 3 || W2->ndim != 3) return 0;
  return moe_plan(T, topk, *W1, *W2, opts ? *opts : kDefaultOpts).total;
}

int mx_moe_forward(const mx_tensor* X, const mx_tensor* Xs, const mx_tensor* W1, const mx_tensor* W1s,
                   const mx_tensor* W2, const mx_tensor* W2s, const float* topk_weights, const void* topk_ids,
                   int32_t ids64, int32_t topk, mx_tensor* out, int32_t scale_mode, const mx_gemm_opts* opts,
                   void* workspace, int64_t workspace_bytes, void* stream) {
  const mx_gemm_opts& o = opts ? *opts : kDefaultOpts;
  if (int rc = check_tensor(X, "X", 2, 2)) return rc;
  if (int rc = check_tensor(Xs, "X_scale", 2, 2)) return rc;
  if (int rc = check_tensor(W1, "W1", 3, 3)) return rc;
  if (int rc = check_tensor(W1s, "W1_scale", 3, 3)) return rc;
  if (int rc = check_tensor(W2, "W2", 3, 3)) return rc;
  if (int rc = check_tensor(W2s, "W2_scale", 3, 3)) return rc;
  if (int rc = check_tensor(out, "out", 2, 2)) return rc;
  if (!topk_weights || !topk_ids) return set_error(MX_ERR_INVALID, "null routing arrays");
  const int64_t T = X->shape[0], H = X->shape[1], E = W1->shape[0], F = W1->shape[1] / 2, H_out = W2->shape[1];
  if (topk <= 0) return set_error(MX_ERR_INVALID, "topk must be positive");
  if (W1->shape[1] % 2 != 0 || W1->shape[2] != H || W2->shape[0] != E || W2->shape[2] != F)
    return set_error(MX_ERR_SHAPE, "W1 must be [E, 2F, H] and W2 [E, H_out, F]");
  if (out->shape[0] != T || out->shape[1] != H_out) return set_error(MX_ERR_SHAPE, "out must be [T, H_out]");
  if (X->dtype != MX_E4M3 || W1->dtype != W2->dtype || (W1->dtype != MX_E4M3 && W1->dtype != MX_E2M1) ||
      Xs->dtype != MX_E8M0 || W1s->dtype != MX_E8M0 || W2s->dtype != MX_E8M0)
    return set_error(MX_ERR_DTYPE, "mx_moe_forward takes E4M3 activations and E4M3 or E2M1 weights with E8M0 scales");
  if (out->dtype != MX_F32 && out->dtype != MX_BF16) return set_error(MX_ERR_DTYPE, "out must be MX_F32 or MX_BF16");
  if (scale_mode != 0 && scale_mode != 1) return set_error(MX_ERR_INVALID, "scale_mode must be 0 (ceil) or 1 (floor)");
  if (H % 32 != 0 || F % 32 != 0 || E <= 0 || T * topk >= 0x7FFFFFFF)
    return set_error(MX_ERR_SHAPE, "H and F must be multiples of 32");
  if (Xs->shape[0] != T || Xs->shape[1] != H / 32) return set_error(MX_ERR_SHAPE, "X_scale must be [T, H/32]");
  if (T == 0 || H_out == 0) return MX_OK;
  // every condition under which one of the steps below could refuse its operands, before anything is enqueued
  auto weights_issue = [&](const mx_tensor* W, const mx_tensor* Ws, int32_t layout) -> const char* {
    if (W->dtype == MX_E2M1 && W->packed_dim != 2) return "FP4 weights are not packed along K";
    if (const char* why = mfma_operand_issue(W->ptr, W->shape[1], W->shape[2], W->stride[1], W->stride[2], W->dtype, 1)) return why;
    if (W->stride[0] % 16 != 0) return "expert pitch of W is not a multiple of 16 bytes";
    if (E * mx_packed_scale_bytes(W->shape[1], W->shape[2]) >= ((int64_t)1 << 31)) return "the packed scales span 2 GiB or more";
    if (layout == MX_SCALE_NATIVE) return ((uintptr_t)Ws->ptr) % 16 != 0 ? "packed scales are not 16-byte aligned" : nullptr;
    if (layout != MX_SCALE_2D) return "scale layout";
    if (Ws->shape[0] != E || Ws->shape[1] != W->shape[1] || Ws->shape[2] != W->shape[2] / 32) return "W_scale must be [E, rows, K/32]";
    if (Ws->stride[2] != 1 || Ws->stride[1] % 4 != 0 || Ws->stride[0] % 4 != 0 || ((uintptr_t)Ws->ptr) % 4 != 0 ||
        W->shape[1] * Ws->stride[1] >= ((int64_t)1 << 31))
      return "W_scale rows are not contiguous and 4-byte aligned";
    return nullptr;
  };
  const char* why = mfma_operand_issue(X->ptr, T, H, X->stride[0], X->stride[1], X->dtype, 1);
  if (!why) why = weights_issue(W1, W1s, o.a_scale_layout);
  if (!why) why = weights_issue(W2, W2s, o.b_scale_layout);
  if (!why && (Xs->stride[1] != 1 || Xs->stride[0] % 4 != 0 || ((uintptr_t)Xs->ptr) % 4 != 0)) why = "X_scale rows are not contiguous and 4-byte aligned";
  if (!why && T * Xs->stride[0] >= ((int64_t)1 << 31)) why = "X_scale spans 2 GiB or more";   // 32-bit lane offsets
  if (!why && (out->stride[1] != 1 || out->stride[0] != H_out)) why = "out is not contiguous";
  if (!why && 2 * F <= 128) why = "F is too small";
  if (!why && H_out <= 128) why = "H_out is too small";
  if (why) return set_error(MX_ERR_LAYOUT, "mx_moe_forward: %s", why);
  MoePlan p = moe_plan(T, topk, *W1, *W2, o);
  // ranges of K are optional: fewer copies can ask for more of them than more copies do, and the room may have been laid out for the latter
  while (p.splits > 1 && workspace_bytes < p.total) p = moe_plan(T, topk, *W1, *W2, o, p.splits - 1);
  if (!p.stream && !p.tiles && p.tile_m % 128 != 0) return set_error(MX_ERR_LAYOUT, "mx_moe_forward: tile_m is not a multiple of 128");
  if (p.n * p.F >= ((int64_t)1 << 31)) return set_error(MX_ERR_LAYOUT, "mx_moe_forward: the activation spans 2 GiB or more");
  if (!workspace || workspace_bytes < p.total)
    return set_error(MX_ERR_WORKSPACE, "workspace of %lld bytes required, %lld given", (long long)p.total, (long long)workspace_bytes);
  if (((uintptr_t)workspace) % 256 != 0) return set_error(MX_ERR_WORKSPACE, "workspace must be 256-byte aligned");
  uint8_t* const ws = (uint8_t*)workspace;
  hipStream_t st = (hipStream_t)stream;

  if (p.stream) {
    MoeStreamArgs a = {};
    a.ids = topk_ids; a.ids64 = ids64; a.n_ids = (int32_t)p.n; a.E = (int32_t)E;
    a.w_fmt = W1->dtype; a.scale_mode = scale_mode;
    a.X = (const uint8_t*)X->ptr; a.Xs = (const uint8_t*)Xs->ptr; a.ldx = X->stride[0]; a.ldxs = Xs->stride[0];
    a.x_rows = (int32_t)T; a.replicas = topk;
    a.W = (const uint8_t*)W1->ptr; a.ldw = W1->stride[1]; a.w_es = W1->stride[0];
    a.Ws = (const uint8_t*)W1s->ptr; a.ws_packed = o.a_scale_layout == MX_SCALE_NATIVE;
    a.ldws = W1s->stride[1]; a.ws_es = a.ws_packed ? mx_packed_scale_bytes(2 * F, H) : W1s->stride[0];
    a.N = (int32_t)(2 * F); a.K = (int32_t)H; a.F = (int32_t)F;
    a.q = ws + p.q; a.qs = ws + p.qs;
    if (int rc = launch_moe_stream(a, true, st)) return rc;
    a.X = ws + p.q; a.Xs = ws + p.qs; a.ldx = F; a.ldxs = F / 32;
    a.x_rows = (int32_t)p.n; a.replicas = 1;
    a.W = (const uint8_t*)W2->ptr; a.ldw = W2->stride[1]; a.w_es = W2->stride[0];
    a.Ws = (const uint8_t*)W2s->ptr; a.ws_packed = o.b_scale_layout == MX_SCALE_NATIVE;
    a.ldws = W2s->stride[1]; a.ws_es = a.ws_packed ? mx_packed_scale_bytes(H_out, F) : W2s->stride[0];
    a.N = (int32_t)H_out; a.K = (int32_t)F;
    a.weights = topk_weights; a.C = (float*)(ws + p.c3);
    if (int rc = launch_moe_stream(a, false, st)) return rc;
  } else if (p.tiles) {
    MoeTileArgs a = {};
    MoeTile* const tiles = (MoeTile*)(ws + p.info);
    int32_t* const slots = (int32_t*)(ws + p.slots);
    if (int rc = launch_moe_tiles(topk_ids, ids64, p.n, (int)E, p.tile_m, tiles, slots, p.max_tiles, st)) return rc;
    a.tiles = tiles; a.slots = slots; a.max_tiles = (int32_t)p.max_tiles; a.tile_rows = p.tile_m;
    a.n_ids = (int32_t)p.n; a.E = (int32_t)E;
    a.w_fmt = W1->dtype; a.scale_mode = scale_mode;
    a.X = (const uint8_t*)X->ptr; a.Xs = (const uint8_t*)Xs->ptr; a.ldx = X->stride[0]; a.ldxs = Xs->stride[0];
    a.x_rows = (int32_t)T; a.replicas = topk;
    a.W = (const uint8_t*)W1->ptr; a.ldw = W1->stride[1]; a.w_es = W1->stride[0];
    a.Ws = (const uint8_t*)W1s->ptr; a.ws_es = mx_packed_scale_bytes(2 * F, H);
    a.N = (int32_t)(2 * F); a.K = (int32_t)H; a.F = (int32_t)F; a.splits = 1;
    a.q = ws + p.q; a.qs = ws + p.qs;
    if (int rc = launch_moe_tile(a, true, st)) return rc;
    a.X = ws + p.q; a.Xs = ws + p.qs; a.ldx = F; a.ldxs = F / 32;
    a.x_rows = (int32_t)p.n; a.replicas = 1;
    a.W = (const uint8_t*)W2->ptr; a.ldw = W2->stride[1]; a.w_es = W2->stride[0];
    a.Ws = (const uint8_t*)W2s->ptr; a.ws_es = mx_packed_scale_bytes(H_out, F);
    a.N = (int32_t)H_out; a.K = (int32_t)F; a.splits = p.splits;
    a.C = (float*)(ws + p.c3); a.c_split = p.n * H_out;
    if (int rc = launch_moe_tile(a, false, st)) return rc;
    return launch_moe_combine(a.C, p.splits, a.c_split, topk_weights, topk_ids, ids64, (int)E, T, topk, H_out, out->ptr, out->dtype, st);
  } else {
    int32_t* const slots = (int32_t*)(ws + p.slots);
    int32_t* const blocks = (int32_t*)(ws + p.blocks);
    // max_slots is what the worst routing needs; the GEMMs walk the tiles of the slots in use only (4096 tokens x 2, 8
    // experts: 36 tile rows, not 39, so 16 rounds of 256 tiles for the first projection where there were 18)
    int32_t* const in_use = (int32_t*)(ws + p.in_use);
    if (int rc = launch_moe_align(topk_ids, ids64, p.n, (int32_t)E, p.tile_m, slots, blocks, in_use, p.max_slots,
                                  (int32_t*)(ws + p.align), st))
      return rc;
    mx_gemm_opts g = kDefaultOpts;
    g.b_scale_layout = o.a_scale_layout;
    mx_tensor c1 = tensor2d(ws + p.c1, MX_BF16, p.n, 2 * F, 2 * F);
    if (int rc = gemm_grouped_impl(X, Xs, W1, W1s, &c1, nullptr, slots, p.max_slots, in_use, blocks, p.tile_m, topk, p.n, &g, ws + p.grouped,
                                 p.grouped_bytes, stream))
      return rc;
    mx_tensor q = tensor2d(ws + p.q, MX_E4M3, p.n, F, F), qs = tensor2d(ws + p.qs, MX_E8M0, p.n, F / 32, F / 32);
    if (int rc = mx_silu_mul_quantize(&c1, &q, &qs, scale_mode, stream)) return rc;
    g.b_scale_layout = o.b_scale_layout;
    mx_tensor c3 = tensor2d(ws + p.c3, MX_F32, p.n, H_out, H_out);
    if (int rc = gemm_grouped_impl(&q, &qs, W2, W2s, &c3, topk_weights, slots, p.max_slots, in_use, blocks, p.tile_m, 1, p.n, &g,
                                 ws + p.grouped, p.grouped_bytes, stream))
      return rc;
  }
  return launch_moe_combine((const float*)(ws + p.c3), 1, 0, nullptr, topk_ids, ids64, (int)E, T, topk, H_out, out->ptr, out->dtype, st);
}

namespace {
// shared by mx_quantize and mx_silu_mul_quantize; K = quantised row length, `up` null for the plain form
int quantize_common(const mx_tensor* x, const void* up, int64_t K, mx_tensor* xq, mx_tensor* scale,
                    int32_t scale_mode, void* stream) {
  if (int rc = check_tensor(xq, "xq", 2, 2)) return rc;
  if (int rc = check_tensor(scale, "scale", 2, 2)) return rc;
  if (x->dtype != MX_F32 && x->dtype != MX_BF16 && x->dtype != MX_F16)
    return set_error(MX_ERR_DTYPE, "x must be MX_F32, MX_BF16 or MX_F16");
  if (!is_elem(xq->dtype)) return set_error(MX_ERR_DTYPE, "xq must be an MX element format");
  if (scale->dtype != MX_E8M0) return set_error(MX_ERR_DTYPE, "scale must be MX_E8M0");
  if (scale_mode != 0 && scale_mode != 1) return set_error(MX_ERR_INVALID, "scale_mode must be 0 (ceil) or 1 (floor)");
  const int64_t rows = x->shape[0];
  if (K < 32)
    return set_error(MX_ERR_SHAPE,
                     "The requested block size 32 is larger than the inner most dimension of the input tensor %lld",
                     (long long)K);
  const int64_t Kpad = (K + 31) / 32 * 32;
  if (xq->shape[0] != rows || xq->shape[1] != Kpad || scale->shape[0] != rows || scale->shape[1] != Kpad / 32)
    return set_error(MX_ERR_SHAPE, "xq must be [rows, %lld] and scale [rows, %lld]", (long long)Kpad,
                     (long long)(Kpad / 32));
  if (x->stride[1] != 1 || xq->stride[1] != 1 || scale->stride[1] != 1)
    return set_error(MX_ERR_LAYOUT, "x, xq and scale must be contiguous along the last axis");
  if (xq->dtype == MX_E2M1 && xq->packed_dim != 1) return set_error(MX_ERR_LAYOUT, "xq must be packed along K");
  QuantArgs q = {};
  q.x = x->ptr; q.xq = (uint8_t*)xq->ptr; q.scale = (uint8_t*)scale->ptr;
  q.rows = rows; q.K = K; q.Kpad = Kpad;
  q.x_ld = x->stride[0]; q.xq_ld = xq->stride[0]; q.sc_ld = scale->stride[0];
  q.x_dtype = x->dtype; q.fmt = xq->dtype; q.scale_mode = scale_mode;
  q.up = up;
  return launch_quantize(q, (hipStream_t)stream);
}
}  // namespace

int mx_quantize(const mx_tensor* x, mx_tensor* xq, mx_tensor* scale, int32_t scale_mode, void* stream) {
  if (int rc = check_tensor(x, "x", 2, 2)) return rc;
  return quantize_common(x, nullptr, x->shape[1], xq, scale, scale_mode, stream);
}

int mx_silu_mul_quantize(const mx_tensor* gate_up, mx_tensor* xq, mx_tensor* scale, int32_t scale_mode,
                         void* stream) {
  if (int rc = check_tensor(gate_up, "gate_up", 2, 2)) return rc;
  if (gate_up->shape[1] % 2 != 0)
    return set_error(MX_ERR_SHAPE, "gate_up must have an even number of columns (gate | up), got %lld",
                     (long long)gate_up->shape[1]);
  const int64_t F = gate_up->shape[1] / 2;
  const int esz = gate_up->dtype == MX_F32 ? 4 : 2;
  const void* up = (const uint8_t*)gate_up->ptr + F * esz;
  return quantize_common(gate_up, up, F, xq, scale, scale_mode, stream);
}

}  // extern "C"
