// Memory-bound helpers around the block-scaled GEMM: MX quantisation, native scale re-layout and the
// MoE slot alignment.  All integer / byte work; results must be bit-exact.
#include "mx_common.h"
#include "mx_load_once.h"
#include "mx_moe_rules.h"
#include "mx_quant.h"

namespace mx {
namespace {

// ================================================================================================
// MX quantiser (replaces the torch-op chain of block_quantize, test/kernels/kernel_utils.py:38-80)
// ================================================================================================
// The shared exponent and the element codes come from encode_block (mx_quant.h), on bit patterns.

__device__ inline float load_as_f32(const void* p, int64_t i, int dtype) {
  if (dtype == MX_F32) return ((const float*)p)[i];
  if (dtype == MX_BF16) return bf16_to_f32(((const uint16_t*)p)[i]);
  return (float)((const _Float16*)p)[i];
}

// EPL consecutive elements starting at element index i (all of them inside K checked by the caller for `vec`)
template <int EPL>
__device__ inline void load_as_f32_vec(const void* p, int64_t i, int dtype, bool vec, int nvalid, float* v) {
  if (vec && dtype == MX_F32) {
#pragma unroll
    for (int h = 0; h < EPL / 4; ++h) {
      const v4f t = *(const v4f*)((const float*)p + i + 4 * h);
      v[4 * h + 0] = t.x; v[4 * h + 1] = t.y; v[4 * h + 2] = t.z; v[4 * h + 3] = t.w;
    }
  } else if (vec && dtype == MX_BF16) {
    uint32_t t[EPL / 2];
    if constexpr (EPL >= 8) {
#pragma unroll
      for (int h = 0; h < EPL / 8; ++h) {
        const v4i r = *(const v4i*)((const uint16_t*)p + i + 8 * h);
        t[4 * h + 0] = (uint32_t)r.x; t[4 * h + 1] = (uint32_t)r.y; t[4 * h + 2] = (uint32_t)r.z; t[4 * h + 3] = (uint32_t)r.w;
      }
    } else {
      const uint2 r = *(const uint2*)((const uint16_t*)p + i);
      t[0] = r.x; t[1] = r.y;
    }
#pragma unroll
    for (int h = 0; h < EPL / 2; ++h) {
      v[2 * h] = bf16_to_f32((uint16_t)t[h]);
      v[2 * h + 1] = bf16_to_f32((uint16_t)(t[h] >> 16));
    }
  } else {
#pragma unroll
    for (int e = 0; e < EPL; ++e) v[e] = e < nvalid ? load_as_f32(p, i + e, dtype) : 0.f;
  }
}

// Where unit `gid` lives: 32 / EPL consecutive units are one 32-element block, EPL consecutive elements per unit.
struct QuantUnit {
  int64_t row, kb, k0;
  int sub;
  bool live;
};

template <int EPL>
__device__ inline QuantUnit quant_unit(const QuantArgs& q, int64_t gid) {
  constexpr int UPB = 32 / EPL;   // units (lanes) per block
  const int64_t KB = q.Kpad / 32;
  QuantUnit u;
  const int64_t blk = gid / UPB;
  u.sub = (int)(gid % UPB);
  u.live = blk < q.rows * KB;
  if (q.rows * KB < ((int64_t)1 << 31)) {   // uniform: 32-bit division is several times cheaper
    const uint32_t b32 = u.live ? (uint32_t)blk : 0u, kb32 = (uint32_t)KB;
    u.row = b32 / kb32;
    u.kb = b32 - (uint32_t)u.row * kb32;
  } else {
    u.row = u.live ? blk / KB : 0;
    u.kb = u.live ? blk % KB : 0;
  }
  u.k0 = u.kb * 32 + u.sub * EPL;
  return u;
}

// the (at most) EPL input values of a unit; the fused producer applies silu(x) * up
template <int EPL>
__device__ inline void quant_load(const QuantArgs& q, const QuantUnit& u, float* v, float* w) {
#pragma unroll
  for (int e = 0; e < EPL; ++e) v[e] = w[e] = 0.f;
  if (!u.live) return;
  const int64_t base = u.row * q.x_ld + u.k0;
  const int esz = q.x_dtype == MX_F32 ? 4 : 2;
  const int nvalid = q.K - u.k0 >= EPL ? EPL : (q.K > u.k0 ? (int)(q.K - u.k0) : 0);
  // 16-byte loads: fp32 in EPL / 4 pieces, bf16 as one (EPL = 8) or an 8-byte one (EPL = 4)
  const int align = (q.x_dtype == MX_F32 || EPL >= 8) ? 16 : 8;
  const bool vec = nvalid == EPL && q.x_dtype != MX_F16 &&
                   ((((uintptr_t)q.x) | ((uintptr_t)q.up) | (uintptr_t)(q.x_ld * esz)) & (align - 1)) == 0;
  load_as_f32_vec<EPL>(q.x, base, q.x_dtype, vec, nvalid, v);
  if (q.up) load_as_f32_vec<EPL>(q.up, base, q.x_dtype, vec, nvalid, w);
}

template <int EPL>
__device__ inline void quant_store(const QuantArgs& q, const QuantUnit& u, float* v, const float* w) {
  constexpr int UPB = 32 / EPL;
  const bool live = u.live;
  const int64_t row = u.row, kb = u.kb, k0 = u.k0;
  const int sub = u.sub;
  if (q.up) {
    const int nvalid = q.K - k0 >= EPL ? EPL : (q.K > k0 ? (int)(q.K - k0) : 0);
#pragma unroll
    for (int e = 0; e < EPL; ++e) v[e] = (live && e < nvalid) ? silu_mul_f32(v[e], w[e]) : 0.f;
  }
  // amax over the block on |bits| (monotone in |x| for finite values; NaN patterns compare largest)
  uint32_t am = 0;
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    const uint32_t a = __builtin_bit_cast(uint32_t, v[e]) & 0x7FFFFFFFu;
    am = a > am ? a : am;
  }
#pragma unroll
  for (int d = 1; d < UPB; d <<= 1) {
    const uint32_t o = (uint32_t)__shfl_xor((int)am, d);
    am = o > am ? o : am;
  }

  uint32_t code[EPL];
  uint8_t scale_byte;
  encode_block<EPL>(v, am, q.fmt, q.scale_mode, code, scale_byte);
  if (!live) return;
  if (q.fmt == MX_E2M1) {
    // low nibble = even element (test/test_mma_scaled.py:155-160)
    uint8_t* out = q.xq + row * q.xq_ld + (k0 >> 1);
    constexpr int NB = EPL / 2;   // output bytes
    uint32_t word[(NB + 3) / 4] = {};
#pragma unroll
    for (int e = 0; e < NB; ++e) word[e / 4] |= (code[2 * e] | (code[2 * e + 1] << 4)) << (8 * (e % 4));
    if (NB >= 4 && ((((uintptr_t)q.xq) | (uintptr_t)q.xq_ld) & (NB - 1)) == 0) {
      if constexpr (NB == 8) *(uint2*)out = make_uint2(word[0], word[1]);
      else *(uint32_t*)out = word[0];
    } else {
#pragma unroll
      for (int e = 0; e < NB; ++e) out[e] = (uint8_t)(word[e / 4] >> (8 * (e % 4)));
    }
  } else {
    uint8_t* out = q.xq + row * q.xq_ld + k0;
    uint32_t word[EPL / 4];
#pragma unroll
    for (int h = 0; h < EPL / 4; ++h)
      word[h] = code[4 * h] | (code[4 * h + 1] << 8) | (code[4 * h + 2] << 16) | (code[4 * h + 3] << 24);
    if ((((((uintptr_t)q.xq) | (uintptr_t)q.xq_ld) & (EPL - 1))) == 0) {
      if constexpr (EPL == 16) *(uint4*)out = make_uint4(word[0], word[1], word[2], word[3]);
      else if constexpr (EPL == 8) *(uint2*)out = make_uint2(word[0], word[1]);
      else *(uint32_t*)out = word[0];
    } else {
#pragma unroll
      for (int e = 0; e < EPL; ++e) out[e] = (uint8_t)code[e];
    }
  }
  if (sub == 0) q.scale[row * q.sc_ld + kb] = scale_byte;
}

// General quantiser: 32 / EPL lanes per 32-element block, EPL consecutive elements per lane; any pitch, alignment and K.
constexpr int kQuantEpl = 8;    // 16 measured no faster (58 -> 60 us on 8192^2 fp32)
template <int EPL>
__global__ __launch_bounds__(256) void quantize_kernel(const QuantArgs q) {
  const QuantUnit u = quant_unit<EPL>(q, (int64_t)blockIdx.x * 256 + threadIdx.x);
  float v[EPL], w[EPL];
  quant_load<EPL>(q, u, v, w);
  quant_store<EPL>(q, u, v, w);
}

// The quantiser of aligned rows (whole blocks, 16-byte loads, stores of a unit in one piece), with the source type and
// the element format known at compile time.
//
// Bound: one pass over the input and the codes.  The general kernel, which decides types and alignment per element
// group and computes the integer route beside the hardware conversions, was short of loads in flight (86 vector
// registers, two units of 16 bytes per thread) and sent each workgroup's scale bytes out in 16-byte pieces of lines that
// other XCDs' workgroups shared: 8192 x 8192 bf16 -> E4M3 took 44 - 49 us (4.1 - 4.6 TB/s), this one 36.6 (5.5 TB/s), and
// 8192 x 14336 of silu(gate) * up 117 us where it took 161
// (133 with an IEEE division per element: there the vector ALUs are the bound).  Inputs that the Infinity Cache cannot hold
// are loaded and their codes stored non-temporally: 8192 x 8192 36.6 -> 33.6 us (6.0 TB/s).  A wave owns U * 64 consecutive
// units, so that a workgroup writes whole lines of scale bytes, all loads of a thread are requested before the first is used,
// and the blocks the hardware conversion does not serve (zero, subnormal, non-finite or extreme amax) are done again
// by the general code from memory, outside of the loop.
template <int SRC>
__device__ __forceinline__ void quant_unpack(const v4i (&t)[SRC == MX_F32 ? 2 : 1], float (&v)[8]) {
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    if constexpr (SRC == MX_F32) {
      v[h] = __builtin_bit_cast(float, (uint32_t)t[0][h]);   // (the cast makes a value of the element: bit_cast of the
      v[4 + h] = __builtin_bit_cast(float, (uint32_t)t[1][h]);   // element itself reads element 0)
    } else if constexpr (SRC == MX_BF16) {
      v[2 * h] = __builtin_bit_cast(float, (uint32_t)t[0][h] << 16);
      v[2 * h + 1] = __builtin_bit_cast(float, (uint32_t)t[0][h] & 0xFFFF0000u);
    } else {
      v[2 * h] = (float)__builtin_bit_cast(_Float16, (uint16_t)(uint32_t)t[0][h]);
      v[2 * h + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)((uint32_t)t[0][h] >> 16));
    }
  }
}

// ONCE: the input is loaded non-temporally (mx_load_once.h); the codes are stored as ever, for the product that reads them next.
template <int SRC, int FMT, bool UP, int U, bool ONCE>
__global__ __launch_bounds__(256) void quantize_rows_kernel(const QuantArgs q) {
  constexpr int NL = SRC == MX_F32 ? 2 : 1;          // 16-byte loads per unit of 8 elements
  constexpr int ESZ = SRC == MX_F32 ? 4 : 2;
  typedef short s2 __attribute__((ext_vector_type(2)));
  typedef uint32_t u2 __attribute__((ext_vector_type(2)));
  auto load = [](const v4i* p) {
    if constexpr (ONCE) return __builtin_nontemporal_load(p);
    else return *p;
  };
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t units = (uint32_t)(q.rows * (q.K / 8)), upr = (uint32_t)(q.K / 8);   // (below 2^31: the launcher's rule)
  const uint32_t first = ((uint32_t)blockIdx.x * 4 + wave) * (U * 64);
  const bool flat = q.x_ld == q.K && q.xq_ld == (FMT == MX_E2M1 ? q.K / 2 : q.K) && q.sc_ld == q.K / 32;   // uniform
  v4i t[U][NL], t2[UP ? U : 1][NL];
  uint32_t row[U], col[U];                           // of a unit; flat: row 0, col = unit
  bool live[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t id = first + u * 64 + lane;
    live[u] = id < units;
    col[u] = live[u] ? id : 0;
    row[u] = 0;
    if (!flat) {
      row[u] = col[u] / upr;
      col[u] -= row[u] * upr;
    }
    const int64_t at = ((int64_t)row[u] * q.x_ld + (int64_t)col[u] * 8) * ESZ;
#pragma unroll
    for (int h = 0; h < NL; ++h) {
      t[u][h] = load((const v4i*)((const uint8_t*)q.x + at + 16 * h));
      if constexpr (UP) t2[u][h] = load((const v4i*)((const uint8_t*)q.up + at + 16 * h));
    }
  }
  const bool floor_mode = q.scale_mode != 0;
  constexpr int EMAX = FMT == MX_E4M3 ? 8 : FMT == MX_E5M2 ? 15 : 2;
  constexpr float FMAX = FMT == MX_E4M3 ? 448.0f : 57344.0f;
  uint32_t again = 0;                                // bit u: unit u's block takes the general route
#pragma unroll
  for (int u = 0; u < U; ++u) {
    float v[8];
    quant_unpack<SRC>(t[u], v);
    if constexpr (UP) {
      float w[8];
      quant_unpack<SRC>(t2[u], w);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = silu_mul_f32(v[e], w[e]);
    }
    uint32_t am = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t a = __builtin_bit_cast(uint32_t, v[e]) & 0x7FFFFFFFu;
      am = a > am ? a : am;
    }
    // the block's other three lanes: quad permutes
    uint32_t o = (uint32_t)__builtin_amdgcn_mov_dpp((int)am, 0xB1, 0xF, 0xF, true);   // lanes 1 0 3 2
    am = o > am ? o : am;
    o = (uint32_t)__builtin_amdgcn_mov_dpp((int)am, 0x4E, 0xF, 0xF, true);            // lanes 2 3 0 1
    am = o > am ? o : am;
    int se;
    if (floor_mode) {
      se = (int)(am >> 23) - 127 - EMAX;
    } else {
      const uint32_t tb = __builtin_bit_cast(uint32_t, fmaxf(__fdiv_rn(__builtin_bit_cast(float, am), 448.0f), 1e-12f));
      se = (int)(tb >> 23) - 127 + ((tb & 0x7FFFFFu) ? 1 : 0);
    }
    const bool fast = am >= 0x00800000u && am < 0x7F800000u && se > -127 && se < 120;
    if (live[u] && !fast) again |= 1u << u;
    const float sc = __builtin_bit_cast(float, (uint32_t)(se + 127) << 23);
    if (FMT != MX_E2M1 && floor_mode) {              // saturating: clamped first, which is exact
      const float lim = __fmul_rn(FMAX, sc);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = __builtin_amdgcn_fmed3f(v[e], -lim, lim);
    }
    if (live[u] && fast) {
      const int64_t block = (int64_t)row[u] * q.sc_ld + col[u] / 4;
      if constexpr (FMT == MX_E2M1) {
        uint32_t r = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, v[0], v[1], sc, 0);
        r = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(r, v[2], v[3], sc, 1);
        r = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(r, v[4], v[5], sc, 2);
        r = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(r, v[6], v[7], sc, 3);
        *(uint32_t*)(q.xq + (int64_t)row[u] * q.xq_ld + (int64_t)col[u] * 4) = r;
      } else {
        uint32_t w[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          s2 r = {0, 0};
          if constexpr (FMT == MX_E4M3) {
            r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, v[4 * h + 0], v[4 * h + 1], sc, false);
            r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, v[4 * h + 2], v[4 * h + 3], sc, true);
          } else {
            r = __builtin_amdgcn_cvt_scalef32_pk_bf8_f32(r, v[4 * h + 0], v[4 * h + 1], sc, false);
            r = __builtin_amdgcn_cvt_scalef32_pk_bf8_f32(r, v[4 * h + 2], v[4 * h + 3], sc, true);
          }
          w[h] = __builtin_bit_cast(uint32_t, r);
        }
        *(u2*)(q.xq + (int64_t)row[u] * q.xq_ld + (int64_t)col[u] * 8) = (u2){w[0], w[1]};
      }
      if ((lane & 3) == 0) q.scale[block] = (uint8_t)(se + 127);
    }
  }
  // (the four lanes of a block agree on `again`: the exchange inside quant_store stays among them)
  if (again) {
    for (int u = 0; u < U; ++u)
      if (again >> u & 1) {
        const QuantUnit un = quant_unit<8>(q, (int64_t)first + u * 64 + lane);
        float v[8], w[8];
        quant_load<8>(q, un, v, w);
        quant_store<8>(q, un, v, w);
      }
  }
}

// ================================================================================================
// Native scale re-layout (see mx_common.h for the layout)
// ================================================================================================
// One workgroup re-lays out 64 rows x 4 K-quads (64 scale bytes per row) of one operand: the bytes are
// staged in LDS with whichever axis is contiguous in the source mapped to consecutive lanes (16-byte
// loads when alignment allows), then every thread assembles the four dwords of one (quad, lane) and
// writes them with one 16-byte store.  Up to two operands (A and B scales of one GEMM) share a launch.
struct PackPair {
  PackArgs p[2];
  int32_t blocks0;   // workgroups that belong to p[0]
};

__device__ inline int64_t scale_src_offset(const PackArgs& p, int64_t srow, int64_t kb, int64_t KB) {
  if (p.layout == MX_SCALE_SWIZZLE_32_4_4) {
    const int64_t m0 = srow >> 7, m2 = (srow & 127) >> 5, m1 = srow & 31, k0 = kb >> 2, k1 = kb & 3;
    return ((m0 * (KB >> 2) + k0) * 32 + m1) * 16 + m2 * 4 + k1;
  }
  return srow * p.s_row + kb * p.s_kb;
}

// up to kPackListMax plain 2-D scale tensors (the operands of a list of problems) in one launch; the entries are
// kept small so that the table travels as a kernel argument
constexpr int kPackListMax = 64;
struct PackEntry {
  const uint8_t* src; uint32_t* dst;
  int64_t rows, K, s_row, s_kb;
  int32_t target;
};
struct PackList {
  PackEntry p[kPackListMax];
  int32_t first_block[kPackListMax + 1];   // workgroups [first_block[i], first_block[i + 1]) belong to p[i]
  int32_t n;
};

__device__ inline void pack_scales_block(const PackArgs& p, const int64_t blk) {
  constexpr int LD = 68;   // LDS row pitch (bytes): 64 scale bytes + 4 so that rows start on distinct banks
  __shared__ __attribute__((aligned(16))) uint8_t tile[64 * LD];
  const int64_t KB = p.K / 32;
  const int64_t KQ = packed_scale_quads(p.K);
  const int64_t qgroups = (KQ + 3) / 4, rgroups = (p.rows + 63) / 64;
  const int64_t b = blk / (qgroups * rgroups);
  const int64_t t64 = (blk / qgroups) % rgroups;
  const int64_t Q0 = (blk % qgroups) * 4;
  const int tid = threadIdx.x;
  const uint8_t* src = p.src + b * p.s_batch;
  const int64_t row0 = t64 * 64, kb0 = Q0 * 16;

  // ---- stage 64 rows x 64 scale bytes; 127 (1.0) wherever the source has nothing -------------------------
  const bool plain = p.layout == MX_SCALE_2D && !p.gather_ids;
  if (plain && p.s_row == 1 && p.s_kb != 1) {
    // rows contiguous in the source: thread = (kb, 16 consecutive rows)
    const int kbi = tid >> 2, c = tid & 3;
    const int64_t kb = kb0 + kbi, r0 = row0 + c * 16;
    alignas(16) uint8_t v[16];
    const uint8_t* s = src + kb * p.s_kb + r0;
    if (kb < KB && r0 + 16 <= p.rows && (((uintptr_t)s) & 15) == 0) {
      *(uint4*)v = *(const uint4*)s;
    } else {
      for (int e = 0; e < 16; ++e) v[e] = (kb < KB && r0 + e < p.rows) ? s[e] : 127;
    }
    for (int e = 0; e < 16; ++e) tile[(c * 16 + e) * LD + kbi] = v[e];
  } else {
    // thread = (row, 16 consecutive K blocks)
    const int rowi = tid >> 2, c = tid & 3;
    const int64_t row = row0 + rowi, kb = kb0 + c * 16;
    int64_t srow = row;
    bool ok = row < p.rows;
    if (p.gather_ids) {
      const int id = ok ? p.gather_ids[row] : -1;
      ok = ok && id >= 0 && id < p.num_valid_ids;
      srow = id / p.replicas;
    }
    alignas(16) uint8_t v[16];
    const uint8_t* s = src + srow * p.s_row + kb;
    if (ok && p.layout == MX_SCALE_2D && p.s_kb == 1 && kb + 16 <= KB && (((uintptr_t)s) & 15) == 0) {
      *(uint4*)v = *(const uint4*)s;
    } else {
      for (int e = 0; e < 16; ++e) v[e] = (ok && kb + e < KB) ? src[scale_src_offset(p, srow, kb + e, KB)] : 127;
    }
    *(uint4*)(tile + rowi * LD + c * 16) = *(const uint4*)v;
  }
  __syncthreads();

  // ---- assemble: thread = (quad q of the group, lane): the 4 x 4 bytes (row, K-step) of the lane, K block
  // (4 (Q0 + q) + t) * 4 + lane / 16 for K-step t; which rows and which index is the dword depend on the target ---
  const int q = tid >> 6, lane = tid & 63, r = lane & 15, g = lane >> 4;
  if (Q0 + q >= KQ) return;
  uint32_t out[4];
  if (p.target == kPackTile32) {
    for (int i4 = 0; i4 < 4; ++i4) {
      const uint8_t* t = tile + (i4 * 16 + r) * LD + q * 16 + g;
      out[i4] = (uint32_t)t[0] | ((uint32_t)t[4] << 8) | ((uint32_t)t[8] << 16) | ((uint32_t)t[12] << 24);
    }
  } else {
    int row[4];
    for (int b = 0; b < 4; ++b) row[b] = p.target == kPackB ? bperm_row(b, r) : 16 * b + r;
    for (int t = 0; t < 4; ++t) {
      const uint8_t* c = tile + q * 16 + 4 * t + g;
      out[t] = (uint32_t)c[row[0] * LD] | ((uint32_t)c[row[1] * LD] << 8) | ((uint32_t)c[row[2] * LD] << 16) |
               ((uint32_t)c[row[3] * LD] << 24);
    }
  }
  uint32_t* dst = p.dst + b * packed_scale_dwords(p.rows, p.K) + ((t64 * KQ + Q0 + q) * 64 + lane) * 4;
  *(uint4*)dst = make_uint4(out[0], out[1], out[2], out[3]);
}

__global__ __launch_bounds__(256) void pack_scales_kernel(const PackPair pp) {
  const bool second = (int)blockIdx.x >= pp.blocks0;
  pack_scales_block(second ? pp.p[1] : pp.p[0], second ? blockIdx.x - pp.blocks0 : blockIdx.x);
}

__global__ __launch_bounds__(256) void pack_scales_list_kernel(const PackList pl) {
  int i = 0;
  while (i + 1 < pl.n && (int)blockIdx.x >= pl.first_block[i + 1]) ++i;   // uniform per workgroup
  const PackEntry& e = pl.p[i];
  PackArgs p = {};
  p.src = e.src; p.dst = e.dst; p.rows = e.rows; p.K = e.K; p.s_row = e.s_row; p.s_kb = e.s_kb;
  p.target = e.target;
  p.layout = MX_SCALE_2D; p.batch = 1; p.replicas = 1;
  pack_scales_block(p, (int)blockIdx.x - pl.first_block[i]);
}

// ================================================================================================
// MoE slot alignment (replaces moe_align_tile_size_torch, test/kernels/fused_moe.py:113-173)
// ================================================================================================
// A stable counting sort of the flattened expert ids; up to 16384 ids and 256 experts in one workgroup (moe_align_one_kernel, below),
// beyond over several, without atomics on global memory and without any slot written twice.  The ids are cut into B contiguous chunks, one per workgroup.
// (The ids may be int64: id_shift = 1 reads their low halves.)
//   moe_hist_kernel (only when B > 1): workgroup b counts the ids of every expert in chunk b -> counts[b][e].
//   moe_place_kernel: workgroup b
//     1. sums column e of `counts` (thread e): ids of expert e in all chunks (total) and in the chunks before
//        its own (base); with B == 1 the totals come from its own counting pass instead;
//     2. exclusive scan of the tile-padded totals over the experts -> first slot of every expert (start);
//     3. places the ids of its chunk in order at start[e] + base[e] + (rank inside the chunk).  Up to 256
//        experts: every thread owns a contiguous segment of the chunk, per-thread per-expert counts live in
//        LDS as u16 (a chunk holds at most 65535 ids, so neither a count nor a prefix inside the chunk can
//        wrap) and become exclusive prefixes over the threads, which is what makes the order stable; more
//        experts: wave 0 walks the chunk 64 ids at a time and ranks equal experts with ballots;
//     4. experts b, b + B, ... : sentinel into the padding behind the expert's ids, expert id into its blocks;
//        all workgroups together: sentinel / expert 0 into the unused tail of the worst-case-sized outputs.
constexpr int kAlignThreads = 256;
constexpr int kAlignSegExperts = 256;      // up to this many experts the segment placement is used
constexpr int64_t kAlignMaxChunk = 65535;  // ids per workgroup (u16 prefixes inside a chunk)

__global__ __launch_bounds__(kAlignThreads) void moe_hist_kernel(const int32_t* __restrict__ topk_ids, int id_shift, int64_t n,
                                                                 int32_t E, int64_t chunk,
                                                                 int32_t* __restrict__ counts) {
  extern __shared__ int32_t sh[];   // [E]
  const int tid = threadIdx.x;
  for (int e = tid; e < E; e += kAlignThreads) sh[e] = 0;
  __syncthreads();
  const int64_t lo = (int64_t)blockIdx.x * chunk, hi = lo + chunk < n ? lo + chunk : n;
  for (int64_t i = lo + tid; i < hi; i += kAlignThreads) {
    const int e = topk_ids[i << id_shift];
    if (e >= 0 && e < E) atomicAdd(&sh[e], 1);
  }
  __syncthreads();
  for (int e = tid; e < E; e += kAlignThreads) counts[(int64_t)blockIdx.x * E + e] = sh[e];
}

__global__ __launch_bounds__(kAlignThreads) void moe_place_kernel(const int32_t* __restrict__ topk_ids, int id_shift, int64_t n,
                                                                  int32_t E, int32_t tile_m, int64_t chunk,
                                                                  const int32_t* __restrict__ counts,
                                                                  int32_t* __restrict__ sorted_ids,
                                                                  int32_t* __restrict__ expert_ids,
                                                                  int32_t* __restrict__ num_slots_out,
                                                                  int64_t max_slots) {
  constexpr int T = kAlignThreads, LD = T + 2;   // row pitch 129 dwords: rows start on consecutive LDS banks
  extern __shared__ int32_t sh[];
  int32_t* total = sh;                  // [E] ids per expert
  int32_t* base = sh + E;               // [E] ids of the expert in earlier chunks; later the write cursor
  int32_t* start = sh + 2 * E;          // [E + 1] first slot of each expert
  int32_t* part = sh + 3 * E + 1;       // [T] partial sums of the scan
  uint16_t* cnt = (uint16_t*)(sh + 3 * E + 1 + T);   // [E][LD], segment placement only
  const int tid = threadIdx.x, B = gridDim.x, b = blockIdx.x;
  const bool seg_mode = E <= kAlignSegExperts;
  const int64_t lo = (int64_t)b * chunk, hi = lo + chunk < n ? lo + chunk : n;
  const int64_t seg = (hi - lo + T - 1) / T;
  const int64_t slo = lo + tid * seg < hi ? lo + tid * seg : hi, shi = slo + seg < hi ? slo + seg : hi;

  // ---- 1. totals and bases ------------------------------------------------------------------------------
  if (seg_mode) {
    for (int i = tid; i < E * LD / 2; i += T) ((uint32_t*)cnt)[i] = 0;
    __syncthreads();
    for (int64_t i = slo; i < shi; ++i) {
      const int e = topk_ids[i << id_shift];
      if (e >= 0 && e < E) cnt[e * LD + tid] += 1;
    }
    __syncthreads();
    if (tid < E) {   // row e -> exclusive prefixes over the threads; the row sum is the chunk's count
      uint16_t* row = cnt + tid * LD;
      int32_t run = 0;
      for (int t = 0; t < T; ++t) {
        const int32_t c = row[t];
        row[t] = (uint16_t)run;
        run += c;
      }
      total[tid] = run;
    }
  } else if (B == 1) {
    for (int e = tid; e < E; e += T) total[e] = 0;
    __syncthreads();
    for (int64_t i = lo + tid; i < hi; i += T) {
      const int e = topk_ids[i << id_shift];
      if (e >= 0 && e < E) atomicAdd(&total[e], 1);
    }
  }
  __syncthreads();
  for (int e = tid; e < E; e += T) {
    int32_t pre = 0;
    if (B > 1) {
      int32_t tot = 0;
      for (int bb = 0; bb < B; ++bb) {
        const int32_t c = counts[(int64_t)bb * E + e];
        if (bb < b) pre += c;
        tot += c;
      }
      total[e] = tot;
    }
    base[e] = pre;
  }
  __syncthreads();
  // ---- 2. first slot of every expert: thread t scans experts [t * per, (t + 1) * per) -------------------
  const int per = (E + T - 1) / T;
  {
    int32_t s2 = 0;
    for (int e = tid * per; e < (tid + 1) * per && e < E; ++e) s2 += (total[e] + tile_m - 1) / tile_m * tile_m;
    part[tid] = s2;
  }
  __syncthreads();
  if (tid == 0) {
    int32_t run = 0;
    for (int t = 0; t < T; ++t) {
      const int32_t c = part[t];
      part[t] = run;
      run += c;
    }
    start[E] = run;
    if (b == 0 && num_slots_out) *num_slots_out = run;
  }
  __syncthreads();
  {
    int32_t run = part[tid];
    for (int e = tid * per; e < (tid + 1) * per && e < E; ++e) {
      start[e] = run;
      run += (total[e] + tile_m - 1) / tile_m * tile_m;
    }
  }
  __syncthreads();
  // ---- 3. placement -------------------------------------------------------------------------------------
  if (seg_mode) {
    for (int64_t i = slo; i < shi; ++i) {
      const int e = topk_ids[i << id_shift];
      if (e >= 0 && e < E) {
        const int32_t pos = start[e] + base[e] + cnt[e * LD + tid];
        cnt[e * LD + tid] += 1;
        sorted_ids[pos] = (int32_t)i;
      }
    }
  } else {
    for (int e = tid; e < E; e += T) base[e] += start[e];   // write cursor of this chunk
    __syncthreads();
    if (tid < 64) {
      for (int64_t i0 = lo; i0 < hi; i0 += 64) {
        const int64_t i = i0 + tid;
        int e = i < hi ? topk_ids[i << id_shift] : -1;
        if (e >= E) e = -1;
        bool todo = e >= 0;
        while (__any(todo)) {
          const uint64_t pending = __ballot(todo);
          const int leader = __builtin_ctzll(pending);
          const int e0 = __shfl(e, leader);
          const bool mine = todo && e == e0;
          const uint64_t same = __ballot(mine);
          if (mine) {
            const int rank = __builtin_popcountll(same & ((1ull << tid) - 1ull));
            sorted_ids[base[e0] + rank] = (int32_t)i;
            todo = false;
          }
          if (tid == leader) base[e0] += __builtin_popcountll(same);
          // wave-synchronous: the next iteration's reads of base[] follow this write in program order
          __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
      }
    }
  }
  // ---- 4. padding, block -> expert map, unused tail (trailing blocks name expert 0) -------------------------
  for (int e = b; e < E; e += B) {
    for (int32_t s2 = start[e] + total[e] + tid; s2 < start[e + 1]; s2 += T) sorted_ids[s2] = (int32_t)n;
    for (int32_t s2 = start[e] + tid * tile_m; s2 < start[e + 1]; s2 += T * tile_m) expert_ids[s2 / tile_m] = e;
  }
  const int32_t used = start[E];
  for (int64_t i = used + (int64_t)b * T + tid; i < max_slots; i += (int64_t)B * T) sorted_ids[i] = (int32_t)n;
  for (int64_t blk = used / tile_m + (int64_t)b * T + tid; blk < max_slots / tile_m; blk += (int64_t)B * T)
    expert_ids[blk] = 0;
}

// The same for up to 16384 ids and 256 experts, in one launch of one workgroup.  A wave owns a contiguous part of the ids, up to 16 per
// lane, which stay in registers.  64 of them at a time: a ballot per bit of the expert's number leaves each lane the lanes of its own
// expert, hence its place among them, and an LDS counter per wave and expert adds the steps before.  Thread e then sums the
// waves' counters of expert e, and a scan over the experts gives the first slots.
// Bound: latency, of one dependent round trip to memory and of the ballots (the two kernels above take three round trips, with a launch
// between, and walk 256 counters one by one).  us, two kernels | this one, without the launch that is saved: 1000 ids, 8 experts 10.4 | 4.7
// (one kernel already), 256 experts 59 | 13; 3000 ids, 8 experts 16.8 | 6.6; 8192 ids, 8 experts 15.8 | 10.2, 64 experts 18.1 |
// 11.7, 256 experts 25.7 | 19.9.  The line: moe_align_in_one_workgroup.  (The sorted ids through LDS, so that whole lines are stored: no
// faster, 16384 ids of 8 experts 11.9, of 256 experts 27.8 against 12.7 and 27.2.)
constexpr int kAlignOneThreads = 1024;
__global__ __launch_bounds__(kAlignOneThreads) void moe_align_one_kernel(const int32_t* __restrict__ topk_ids, int id_shift, int n, int E,
                                                                         int tile_m, int32_t* __restrict__ sorted_ids,
                                                                         int32_t* __restrict__ expert_ids,
                                                                         int32_t* __restrict__ num_slots_out, int64_t max_slots,
                                                                         int64_t max_blocks) {
  constexpr int T = kAlignOneThreads, W = T / 64, PER = kAlignOneIds / T;
  __shared__ int32_t count[W][kAlignOneExperts], start[kAlignOneExperts + 1], total[kAlignOneExperts], wave_sum[W];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int steps = (n + T - 1) / T, first = wave * steps * 64 + lane;
  int e[PER], place[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = first + 64 * k;
    e[k] = k < steps && i < n ? topk_ids[(int64_t)i << id_shift] : -1;
    if (e[k] >= E) e[k] = -1;
  }
  for (int x = lane; x < E; x += 64) count[wave][x] = 0;
  __syncthreads();
  const int bits = E > 1 ? 32 - __builtin_clz(E - 1) : 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    if (k >= steps) break;                           // uniform
    const bool valid = e[k] >= 0;
    uint64_t same = __builtin_amdgcn_ballot_w64(valid);
    for (int b = 0; b < bits; ++b) {
      const bool set = e[k] >> b & 1;
      const uint64_t m = __builtin_amdgcn_ballot_w64(set);
      same &= set ? m : ~m;
    }
    const int rank = __builtin_popcountll(same & ((1ull << lane) - 1));
    int before = 0;
    if (valid) before = count[wave][e[k]];
    place[k] = before + rank;
    // wave-synchronous: every lane has read its counter when the first of each expert writes it, and reads the next step's after that
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (valid && rank == 0) count[wave][e[k]] = before + __builtin_popcountll(same);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  __syncthreads();
  int mine = 0;
  if (tid < E) {
    int c[W];
#pragma unroll
    for (int w = 0; w < W; ++w) c[w] = count[w][tid];
#pragma unroll
    for (int w = 0; w < W; ++w) {
      count[w][tid] = mine;
      mine += c[w];
    }
    total[tid] = mine;
  }
  const int padded = (mine + tile_m - 1) / tile_m * tile_m;
  int sum = padded;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(sum, d);
    if (lane >= d) sum += o;
  }
  if (lane == 63) wave_sum[wave] = sum;
  __syncthreads();
  if (tid < E) {
    for (int w = 0; w < wave; ++w) sum += wave_sum[w];
    start[tid] = sum - padded;
    if (tid == E - 1) {
      start[E] = sum;
      if (num_slots_out) *num_slots_out = sum;
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < PER; ++k)
    if (k < steps && e[k] >= 0) sorted_ids[start[e[k]] + count[wave][e[k]] + place[k]] = first + 64 * k;
  // padding, block -> expert map, unused tail (as above)
  for (int x = wave; x < E; x += W) {
    for (int s = start[x] + total[x] + lane; s < start[x + 1]; s += 64) sorted_ids[s] = n;
    for (int b = start[x] / tile_m + lane; b < start[x + 1] / tile_m; b += 64) expert_ids[b] = x;   // (whole tiles)
  }
  const int used = start[E];
  for (int64_t i = used + tid; i < max_slots; i += T) sorted_ids[i] = n;
  for (int64_t blk = used / tile_m + tid; blk < max_blocks; blk += T) expert_ids[blk] = 0;
}

// ================================================================================================
// Split-K reduction: C = sum of the fp32 partial products (analogue of the second pass of
// matmul_split_k_kernel, test/kernels/matmul.py:103-140)
// ================================================================================================
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ part, int splits,
                                                            int64_t M, int64_t N, void* C, int64_t ldc,
                                                            int c_dtype, int accumulate) {
  const int64_t n4 = (N + 3) / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= M * n4) return;
  const int64_t m = i / n4, n = (i % n4) * 4;
  const int cnt = N - n >= 4 ? 4 : (int)(N - n);
  float s[4] = {0.f, 0.f, 0.f, 0.f};
  for (int p = 0; p < splits; ++p) {   // fixed order: results do not depend on scheduling
    const float* src = part + ((int64_t)p * M + m) * N + n;
    if (cnt == 4 && (N & 3) == 0) {
      const v4f t = *(const v4f*)src;
      s[0] += t.x; s[1] += t.y; s[2] += t.z; s[3] += t.w;
    } else {
      for (int e = 0; e < cnt; ++e) s[e] += src[e];
    }
  }
  if (c_dtype == MX_F32) {
    float* c = (float*)C + m * ldc + n;
    for (int e = 0; e < cnt; ++e) c[e] = accumulate ? c[e] + s[e] : s[e];
  } else {
    uint16_t* c = (uint16_t*)C + m * ldc + n;
    for (int e = 0; e < cnt; ++e) c[e] = f32_to_bf16(accumulate ? bf16_to_f32(c[e]) + s[e] : s[e]);
  }
}

}  // namespace

template <int SRC, int FMT>
static hipError_t launch_quantize_rows(const QuantArgs& q, int64_t units, hipStream_t stream) {
  // four units per thread once that leaves every CU several waves per SIMD, else one (a single row is a few waves: the
  // launch is all latency).  The silu form holds two inputs per unit and computes for longer: two.
#define MX_Q(UP, U, ONCE) return launch_kernel(quantize_rows_kernel<SRC, FMT, UP, U, ONCE>, dim3((unsigned)((units + 256 * U - 1) / (256 * U))), dim3(256), 0, stream, q)
  const bool large = units >= ((int64_t)1 << 20);
  if (q.up) { if (large) MX_Q(true, 2, false); else MX_Q(true, 1, false); }
  else if (large) { if (quantize_loads_once(units * 8)) MX_Q(false, 4, true); else MX_Q(false, 4, false); }
  else MX_Q(false, 1, false);
#undef MX_Q
}

int launch_quantize(const QuantArgs& q, hipStream_t stream) {
  const int64_t units = q.rows * (q.Kpad / 32) * (32 / kQuantEpl);
  if (units <= 0) return MX_OK;
  const int64_t blocks = (units + 255) / 256;
  if (blocks > 0x7FFFFFFF) return set_error(MX_ERR_SHAPE, "quantize: tensor too large");
  // whole blocks, rows of x at multiples of 16 bytes, a unit's codes (8 or 4 bytes) aligned
  const int esz = q.x_dtype == MX_F32 ? 4 : 2, cb = q.fmt == MX_E2M1 ? 4 : 8;
  const bool rows_ok = q.K % 32 == 0 && units < ((int64_t)1 << 31) && (((uintptr_t)q.x | (uintptr_t)q.up | (uintptr_t)(q.x_ld * esz)) & 15) == 0 &&
                       (((uintptr_t)q.xq | (uintptr_t)q.xq_ld) & (cb - 1)) == 0;
  hipError_t e = hipSuccess;
  if (rows_ok) {
#define MX_CASE(SRC, FMT) \
    if (q.x_dtype == SRC && q.fmt == FMT) e = launch_quantize_rows<SRC, FMT>(q, units, stream);
    MX_CASE(MX_BF16, MX_E4M3)
    MX_CASE(MX_BF16, MX_E5M2)
    MX_CASE(MX_BF16, MX_E2M1)
    MX_CASE(MX_F32, MX_E4M3)
    MX_CASE(MX_F32, MX_E5M2)
    MX_CASE(MX_F32, MX_E2M1)
    MX_CASE(MX_F16, MX_E4M3)
    MX_CASE(MX_F16, MX_E5M2)
    MX_CASE(MX_F16, MX_E2M1)
#undef MX_CASE
  } else {
    e = launch_kernel(quantize_kernel<kQuantEpl>, dim3((unsigned)blocks), dim3(256), 0, stream, q);
  }
  if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "quantize_kernel launch: %s", hipGetErrorString(e));
  return MX_OK;
}

int launch_pack_scales_pair(const PackArgs* a, const PackArgs* b, hipStream_t stream) {
  PackPair pp = {};
  int64_t blocks[2] = {0, 0};
  const PackArgs* ops[2] = {a, b};
  int n = 0;
  for (int i = 0; i < 2; ++i) {
    const PackArgs* p = ops[i];
    if (!p || p->rows <= 0 || p->K <= 0 || p->batch <= 0) continue;
    pp.p[n] = *p;
    blocks[n] = ((p->rows + 63) / 64) * ((packed_scale_quads(p->K) + 3) / 4) * p->batch;
    ++n;
  }
  if (n == 0) return MX_OK;
  const int64_t total = blocks[0] + blocks[1];
  if (total > 0x7FFFFFFF) return set_error(MX_ERR_SHAPE, "pack_scales: tensor too large");
  pp.blocks0 = (int32_t)blocks[0];
  hipError_t e = launch_kernel(pack_scales_kernel, dim3((unsigned)total), dim3(256), 0, stream, pp);
  if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "pack_scales_kernel launch: %s", hipGetErrorString(e));
  return MX_OK;
}

int launch_pack_scales_list(const PackArgs* list, int n, hipStream_t stream) {
  for (int i0 = 0; i0 < n; i0 += kPackListMax) {
    PackList pl = {};
    int64_t total = 0;
    for (int i = i0; i < n && i < i0 + kPackListMax; ++i) {
      const PackArgs& p = list[i];
      if (p.rows <= 0 || p.K <= 0 || p.batch <= 0) continue;
      if (p.layout != MX_SCALE_2D || p.batch != 1 || p.gather_ids)
        return set_error(MX_ERR_INVALID, "pack_scales list: plain 2-D scale tensors only");
      pl.p[pl.n] = PackEntry{p.src, p.dst, p.rows, p.K, p.s_row, p.s_kb, p.target};
      pl.first_block[pl.n] = (int32_t)total;
      total += ((p.rows + 63) / 64) * ((packed_scale_quads(p.K) + 3) / 4) * p.batch;
      if (total > 0x7FFFFFFF) return set_error(MX_ERR_SHAPE, "pack_scales: tensors too large");
      ++pl.n;
    }
    if (pl.n == 0) continue;
    pl.first_block[pl.n] = (int32_t)total;
    hipError_t e = launch_kernel(pack_scales_list_kernel, dim3((unsigned)total), dim3(256), 0, stream, pl);
    if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "pack_scales_list_kernel launch: %s", hipGetErrorString(e));
  }
  return MX_OK;
}

int launch_pack_scales(const PackArgs& p, hipStream_t stream) {
  return launch_pack_scales_pair(&p, nullptr, stream);
}

int launch_splitk_reduce(const float* partials, int splits, int64_t M, int64_t N, void* C, int64_t ldc,
                         int c_dtype, int accumulate, hipStream_t stream) {
  const int64_t threads = M * ((N + 3) / 4);
  if (threads <= 0) return MX_OK;
  hipError_t e = launch_kernel(splitk_reduce_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, partials,
                               splits, M, N, C, ldc, c_dtype, accumulate);
  if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "splitk_reduce_kernel launch: %s", hipGetErrorString(e));
  return MX_OK;
}

// chunks (= workgroups) the ids are cut into: about 1024 ids each, at most 256 chunks unless a chunk would then
// exceed what the u16 prefixes of the placement hold
void moe_align_plan(int64_t num_ids, int64_t& chunk, int64_t& blocks) {
  chunk = (num_ids + 255) / 256;
  if (chunk < 1024) chunk = 1024;
  if (chunk > kAlignMaxChunk) chunk = kAlignMaxChunk;
  blocks = num_ids > 0 ? (num_ids + chunk - 1) / chunk : 1;
}

int64_t moe_align_workspace_bytes(int64_t num_ids, int32_t num_experts) {
  int64_t chunk, blocks;
  moe_align_plan(num_ids, chunk, blocks);
  return blocks > 1 ? blocks * num_experts * (int64_t)sizeof(int32_t) : 0;
}

int launch_moe_align(const void* ids, int ids64, int64_t num_ids, int32_t num_experts, int32_t tile_m,
                     int32_t* sorted_token_ids, int32_t* sorted_expert_ids, int32_t* num_slots_out,
                     int64_t max_slots, int32_t* counts, hipStream_t stream) {
  int64_t chunk, blocks;
  moe_align_plan(num_ids, chunk, blocks);
  const int32_t* topk_ids = (const int32_t*)ids;
  const int id_shift = ids64 ? 1 : 0;
  if (moe_align_in_one_workgroup(num_ids, num_experts)) {
    hipError_t e = launch_kernel(moe_align_one_kernel, dim3(1), dim3(kAlignOneThreads), 0, stream, topk_ids, id_shift, (int)num_ids, (int)num_experts,
                                 (int)tile_m, sorted_token_ids, sorted_expert_ids, num_slots_out, max_slots, max_slots / tile_m);
    if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "moe_align_one_kernel launch: %s", hipGetErrorString(e));
    return MX_OK;
  }
  const bool seg = num_experts <= kAlignSegExperts;
  const size_t lds = (size_t)(3 * num_experts + 1 + kAlignThreads) * sizeof(int32_t) +
                     (seg ? (size_t)num_experts * (kAlignThreads + 2) * sizeof(uint16_t) : 0);
  if (lds > 150 * 1024) return set_error(MX_ERR_SHAPE, "moe_align: too many experts (%d)", num_experts);
  if (blocks > 0x7FFFFFFF) return set_error(MX_ERR_SHAPE, "moe_align: too many ids");
  static int attr_done = 0;   // benign race: the attribute call is idempotent
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute((const void*)moe_place_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       160 * 1024);
    if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "hipFuncSetAttribute(moe_align): %s", hipGetErrorString(e));
    attr_done = 1;
  }
  if (blocks > 1) {
    hipError_t e = launch_kernel(moe_hist_kernel, dim3((unsigned)blocks), dim3(kAlignThreads), (size_t)num_experts * sizeof(int32_t),
                                 stream, topk_ids, id_shift, num_ids, num_experts, chunk, counts);
    if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "moe_hist_kernel launch: %s", hipGetErrorString(e));
  }
  hipError_t e = launch_kernel(moe_place_kernel, dim3((unsigned)blocks), dim3(kAlignThreads), lds, stream, topk_ids, id_shift, num_ids,
                               num_experts, tile_m, chunk, counts, sorted_token_ids, sorted_expert_ids, num_slots_out, max_slots);
  if (e != hipSuccess) return set_error(MX_ERR_LAUNCH, "moe_place_kernel launch: %s", hipGetErrorString(e));
  return MX_OK;
}

}  // namespace mx
