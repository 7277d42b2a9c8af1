// MX encoding of a 32-element block that several lanes hold together: shared by the quantiser (mx_aux.hip) and by the
// kernels that quantise what they have just computed.
#pragma once
#include "mx_common.h"

namespace mx {

// The shared exponent is computed on bit patterns.  Element conversion has two routes with identical
// results: the gfx950 scaled-conversion instructions for ordinary blocks, and an integer route (value =
// sig * 2^(ex-150) divided by 2^se by subtracting exponents, then rounded to nearest even onto the target
// grid in one step) for blocks with a zero / subnormal amax, inf / NaN or an extreme scale, where denormal
// modes or the instruction's special cases could otherwise change a bit.

struct Unpacked {
  uint32_t sig;   // 24-bit significand with the leading one at bit 23 (0 for zero)
  int ex;         // biased exponent such that value = sig * 2^(ex - 150)
  uint32_t sign;  // 0 or 1
  int cls;        // 0 finite, 1 inf, 2 nan
};

__device__ inline Unpacked unpack_f32(uint32_t bits) {
  Unpacked u;
  u.sign = bits >> 31;
  const uint32_t a = bits & 0x7FFFFFFFu;
  u.cls = a > 0x7F800000u ? 2 : (a == 0x7F800000u ? 1 : 0);
  int ex = (int)(a >> 23);
  uint32_t sig = a & 0x7FFFFFu;
  if (ex == 0) {
    if (sig != 0) {  // subnormal: normalise
      const int lz = __builtin_clz(sig) - 8;
      sig <<= lz;
      ex = 1 - lz;
    }
  } else {
    sig |= 0x800000u;
  }
  u.sig = sig;
  u.ex = ex;
  return u;
}

// round-to-nearest-even of sig / 2^sh, sh in [1, 31]
__device__ inline uint32_t rne_shift(uint32_t sig, int sh) {
  return (sig + ((1u << (sh - 1)) - 1u) + ((sig >> sh) & 1u)) >> sh;
}

// Generic minifloat encoder: MBITS mantissa bits, minimum normal exponent EMIN, exponent bias BIAS.
// Returns the magnitude code without clamping (may exceed the format's largest finite code).
template <int MBITS, int EMIN, int BIAS>
__device__ inline uint32_t encode_mag(const Unpacked& u, int se) {
  if (u.sig == 0) return 0;
  const int E = u.ex - 127 - se;            // exponent of x / 2^se
  const int Eq = E > EMIN ? E : EMIN;
  int sh = (23 - MBITS) + (Eq - E);
  if (sh > 31) sh = 31;                     // anything this small rounds to zero
  const uint32_t n = rne_shift(u.sig, sh);  // in units of 2^(Eq - MBITS); normal range: [2^MBITS, 2^(MBITS+1)]
  if (E > 300) return 0xFFFFu;              // cannot happen for finite fp32 / E8M0 scales; keeps shifts sane
  return (uint32_t)((Eq + BIAS - 1) << MBITS) + n;
}

__device__ inline uint32_t encode_e4m3(const Unpacked& u, int se, bool saturate) {
  const uint32_t s = u.sign << 7;
  if (u.cls == 2) return s | 0x7F;
  if (u.cls == 1) return s | (saturate ? 0x7Eu : 0x7Fu);
  uint32_t c = encode_mag<3, -6, 7>(u, se);
  if (c > 0x7E) c = saturate ? 0x7E : 0x7F;   // torch's cast: above 448 after rounding -> NaN
  return s | c;
}

__device__ inline uint32_t encode_e5m2(const Unpacked& u, int se, bool saturate) {
  const uint32_t s = u.sign << 7;
  if (u.cls == 2) return s | 0x7F;
  if (u.cls == 1) return s | (saturate ? 0x7Bu : 0x7Cu);
  uint32_t c = encode_mag<2, -14, 15>(u, se);
  if (c > 0x7B) c = saturate ? 0x7B : 0x7C;   // IEEE-like: overflow -> inf
  return s | c;
}

__device__ inline uint32_t encode_e2m1(const Unpacked& u, int se) {
  const uint32_t s = u.sign << 3;
  if (u.cls != 0) return s | 7;
  uint32_t c = encode_mag<1, 0, 1>(u, se);
  if (c > 7) c = 7;                           // finite-only format: clamp to +-6
  return s | c;
}

// 1 / d, correctly rounded, for d in [1, 2^126): the hardware's reciprocal and one Newton step in fused arithmetic give the
// bits of the IEEE division for every such d (mx_probe_rcp compares all 2^23 significands of the 126 exponents; from 2^126
// on the result is subnormal and they do not).  3 instructions for 12.
__device__ inline float rcp_rn(float d) {
  const float r = __builtin_amdgcn_rcpf(d);
  return __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
}

// silu(a) * b = a / (1 + exp(-a)) * b as a fixed sequence of correctly rounded fp32 operations (nothing
// contracted, nothing approximate in its result), so that a host restatement with the same sequence gets the
// same bits: exp(-a) = 2^z, z = -a * log2(e) clamped to +-125, z = n + f with n = rint(z), 2^f by the
// degree-7 Taylor polynomial in f * ln 2 (|f| <= 0.5: truncation error below 1e-8), scaled by 2^n exactly.
__device__ inline float silu_mul_f32(float a, float b) {
  float z = __fmul_rn(-a, 1.44269504f);
  z = fminf(fmaxf(z, -125.0f), 125.0f);
  const float n = __builtin_rintf(z);
  const float f = __fsub_rn(z, n);
  float p = 1.52527338e-5f;
  p = __fadd_rn(__fmul_rn(p, f), 1.54035304e-4f);
  p = __fadd_rn(__fmul_rn(p, f), 1.33335581e-3f);
  p = __fadd_rn(__fmul_rn(p, f), 9.61812911e-3f);
  p = __fadd_rn(__fmul_rn(p, f), 5.55041087e-2f);
  p = __fadd_rn(__fmul_rn(p, f), 2.40226507e-1f);
  p = __fadd_rn(__fmul_rn(p, f), 6.93147181e-1f);
  p = __fadd_rn(__fmul_rn(p, f), 1.0f);
  const float e = __fmul_rn(p, __builtin_bit_cast(float, (uint32_t)((int)n + 127) << 23));
  const float s = rcp_rn(__fadd_rn(1.0f, e));             // e is in [2^-125, 2^125]
  const float t = a < -87.5f ? 0.0f : __fmul_rn(a, s);   // exp(-a) is past the clamp: the true value is below 2^-120
  return __fmul_rn(t, b);
}

// Codes of EPL elements of a block whose largest magnitude has the bit pattern `am`, and the block's scale byte.
// scale_mode 0: the reference's ceiling rule, non-saturating; 1: the OCP floor rule, saturating.
template <int EPL>
__device__ inline void encode_block(const float* v, const uint32_t am, const int fmt, const int scale_mode, uint32_t* code,
                                    uint8_t& scale_byte) {
  uint32_t bits[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) bits[e] = __builtin_bit_cast(uint32_t, v[e]);
  // shared exponent
  int se;
  if (scale_mode == 0) {
    // reference rule: 2^ceil(log2(max(amax/448, 1e-12))), ceiling taken exactly on the fp32 quotient
    // (a block with an inf or NaN amax never uses this exponent: see nonfinite_ceil below)
    float t = __fdiv_rn(__builtin_bit_cast(float, am), 448.0f);
    t = t > 1e-12f ? t : 1e-12f;
    const uint32_t tb = __builtin_bit_cast(uint32_t, t);
    se = (int)(tb >> 23) - 127 + ((tb & 0x7FFFFFu) ? 1 : 0);
  } else {
    // OCP MX v1.0: floor(log2 amax) - emax_elem; all-zero block -> smallest scale
    const int emax = fmt == MX_E4M3 ? 8 : (fmt == MX_E5M2 ? 15 : 2);
    if (am == 0) {
      se = -127;
    } else {
      const int ex = (int)(am >> 23);
      const int fl = ex ? ex - 127 : (31 - __builtin_clz(am)) - 149;
      se = fl - emax;
    }
  }
  se = se < -127 ? -127 : (se > 127 ? 127 : se);
  const bool saturate = scale_mode != 0;

  // Reference rule with a non-finite amax: torch.clamp(min=) keeps NaN and inf / 448 stays inf, so the scale is
  // NaN or inf, both of which the cast to float8_e8m0fnu writes as 0xFF; x / scale is then NaN for every
  // element of a NaN block (the element's own sign if it is a NaN itself), and for an inf block NaN where
  // |x| is inf (inf / inf is the default NaN, whose sign bit is set on the hosts the reference runs on) and a
  // signed zero elsewhere.  E2M1 has no NaN: non-finite elements saturate to +-6 as in the finite case.
  const bool nonfinite_ceil = scale_mode == 0 && am >= 0x7F800000u;
  if (nonfinite_ceil) {
    const bool blk_nan = am > 0x7F800000u;
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const uint32_t a = bits[e] & 0x7FFFFFFFu, sgn = bits[e] >> 31;
      if (fmt == MX_E2M1) code[e] = (sgn << 3) | ((blk_nan || a == 0x7F800000u) ? 7u : 0u);
      else if (a > 0x7F800000u) code[e] = (sgn << 7) | 0x7Fu;
      else if (blk_nan) code[e] = 0x7Fu;
      else if (a == 0x7F800000u) code[e] = 0xFFu;
      else code[e] = sgn << 7;
    }
  } else
  // Blocks whose amax is a normal finite number and whose scale 2^se is a normal float take the hardware
  // scaled conversions (v_cvt_scalef32_pk_*: x / 2^se rounded to nearest even; FP8 overflows to NaN / inf,
  // FP4 saturates -- measured on MI355X against the integer encoders below for 270 k inputs per format).
  // The saturating FP8 rule clamps the magnitude to max_normal * 2^se first, which is exact.  Everything
  // else (zero or subnormal amax, inf / NaN, extreme scales) goes through the integer encoders.
  if (am >= 0x00800000u && am < 0x7F800000u && se > -127 && se < 120) {
    typedef short s2 __attribute__((ext_vector_type(2)));
    const float sc = __builtin_bit_cast(float, (uint32_t)(se + 127) << 23);
    float x[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) x[e] = v[e];
    if (saturate && fmt != MX_E2M1) {
      const float lim = __fmul_rn(fmt == MX_E4M3 ? 448.0f : 57344.0f, sc);
#pragma unroll
      for (int e = 0; e < EPL; ++e) x[e] = __builtin_copysignf(fminf(__builtin_fabsf(x[e]), lim), x[e]);
    }
#pragma unroll
    for (int h = 0; h < EPL / 4; ++h) {   // four elements at a time
      uint32_t packed;
      if (fmt == MX_E4M3) {
        s2 r = {0, 0};
        r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, x[4 * h + 0], x[4 * h + 1], sc, false);
        r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, x[4 * h + 2], x[4 * h + 3], sc, true);
        packed = __builtin_bit_cast(uint32_t, r);
      } else if (fmt == MX_E5M2) {
        s2 r = {0, 0};
        r = __builtin_amdgcn_cvt_scalef32_pk_bf8_f32(r, x[4 * h + 0], x[4 * h + 1], sc, false);
        r = __builtin_amdgcn_cvt_scalef32_pk_bf8_f32(r, x[4 * h + 2], x[4 * h + 3], sc, true);
        packed = __builtin_bit_cast(uint32_t, r);
      } else {
        uint32_t r = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, x[4 * h + 0], x[4 * h + 1], sc, 0);
        r = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(r, x[4 * h + 2], x[4 * h + 3], sc, 1);
        packed = (r & 0xFu) | ((r & 0xF0u) << 4) | ((r & 0xF00u) << 8) | ((r & 0xF000u) << 12);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) code[4 * h + e] = (packed >> (8 * e)) & 0xFFu;
    }
  } else {
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const Unpacked un = unpack_f32(bits[e]);
      code[e] = fmt == MX_E4M3 ? encode_e4m3(un, se, saturate)
                : fmt == MX_E5M2 ? encode_e5m2(un, se, saturate)
                                   : encode_e2m1(un, se);
    }
  }
  scale_byte = nonfinite_ceil ? (uint8_t)0xFF : (uint8_t)(se + 127);
}

}  // namespace mx
