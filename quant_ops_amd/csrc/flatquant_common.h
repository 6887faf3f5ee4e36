// Device helpers shared by the quantize kernels: the per-token scale, the code
// of a quotient, MFMA operands and the packed-pair epilogue.
#pragma once

#include <type_traits>

#include "common.h"

namespace qo {

// ---------------------------------------------------------------------------
// Scale and code, shared by the quantize kernels.
// ---------------------------------------------------------------------------

// Per-token scale from the raw (unrounded) fp32 extremes of Y. Rounding to D is
// monotonic, so rnd_D(max y) == max rnd_D(y): this is amax/amin of the D tensor
// (ops.py:108-109), then maximum(|rnd(min*c)|, rnd(max*c)) (ops.py:112), then
// rnd(./7) clamped below by rnd_D(1e-8) (ops.py:113).
template <class DT>
__device__ inline float fq_scale(float ymax_raw, float ymin_raw, float clip) {
  const float hi = DT::round(ymax_raw);
  const float lo = DT::round(ymin_raw);
  const float t_lo = DT::round(lo * clip);
  const float t_hi = DT::round(hi * clip);
  const float bound = fmaxf(fabsf(t_lo), t_hi);
  const float s = DT::round(opaque(bound) / 7.0f);
  return fmaxf(s, DT::round(1e-8f));
}

// The same scale from max |Y| of the D-rounded Y, valid for clip > 0:
// rounding to nearest even is sign-symmetric and monotonic, so
// max(|rnd(rnd(min) c)|, rnd(rnd(max) c)) = rnd(max |rnd(y)| c).
template <class DT>
__device__ inline float fq_scale_abs(float amax, float clip) {
  const float bound = DT::round(amax * clip);
  const float s = DT::round(opaque(bound) / 7.0f);
  return fmaxf(s, DT::round(1e-8f));
}

// Code of one element from its D-rounded quotient t = rnd_D(y / s):
// clamp(round_half_even(t), -8, 7) (ops.py:117). A NaN quotient (0/0 when an
// fp16 token's scale rounds to 0) becomes 0 through the reference's int8 cast
// and nibble 0 (code -8) through its uint8 cast before packing (ops.py:122);
// both are reproduced here.
template <bool PACK>
__device__ inline int fq_code_from_quot(float t) {
  if (t != t) return PACK ? -8 : 0;
  const float c = fminf(fmaxf(t, -8.0f), 7.0f);
  return (int)__builtin_rintf(c);
}

template <class DT>
struct MfmaOps;

// V: 8-element operands of the 16x16x32 MFMA. An odd trailing 16-deep slab of
// the second product (M / 16 odd) is a zero-padded 32-deep slab: elements 0..3
// of lane group g hold k = 4g .. 4g+3 (the rows of Z's accumulator), elements
// 4..7 of both operands are zero, which leaves the MFMA's sum unchanged. (The
// 16x16x16 MFMA gave wrong results in that role on gfx950.)
template <>
struct MfmaOps<F16T> {
  using V = v8h;
  __device__ static inline v4f mfma(V a, V b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

template <>
struct MfmaOps<BF16T> {
  using V = v8bf;
  __device__ static inline v4f mfma(V a, V b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

// Epilogue on packed pairs. A lane's Y values come in pairs (MFMA block h = 0
// and 1 at the same accumulator row r) that belong in nibbles r and r + 4 of
// one output word, so each pair is kept as two 16-bit D values in one VGPR
// (rounding point 2 for both with one v_cvt_pk). Quantizing a pair:
//   a = clamp(y * rcp, -8, 7) in float32   (clamp commutes with the roundings
//                                           below because -8 and 7 are D values)
//   t = rnd_D(a)                           (one v_cvt_pk for the pair)
//   t + magic                              (round half to even to an integer)
// The magic constant leaves q + 8 in the low bits of each result; shifting the
// pair's bits by 4r and adding puts both codes in place, and the constant bits
// the magic leaves above the codes add up to kJunk, removed once per word.
// y * rcp stands in for the fallback's y / s (IEEE): the two differ only when
// the quotient lies within a few float32 ulps of a rounding boundary of D.
template <class DT>
struct FqEpi;

template <>
struct FqEpi<F16T> {
  __device__ static inline uint32_t pack(float a, float b) {
    const v2h h = {(_Float16)opaque(a), (_Float16)opaque(b)};
    return __builtin_bit_cast(uint32_t, h);
  }
  // The same rounding of two MFMA accumulator values. An MFMA result has no
  // product for the compiler to fuse into the conversion, so no opaque() is
  // needed (which would copy accumulators that are read again for the absmax).
  __device__ static inline uint32_t pack_acc(float a, float b) {
    const v2h h = {(_Float16)a, (_Float16)b};
    return __builtin_bit_cast(uint32_t, h);
  }
  __device__ static inline float lo(uint32_t p) { return (float)__builtin_bit_cast(v2h, p)[0]; }
  __device__ static inline float hi(uint32_t p) { return (float)__builtin_bit_cast(v2h, p)[1]; }
  // fp16: 1544 = 1536 + 8 has a unit ulp, so t + 1544 is the integer 1536 + q + 8,
  // bits 0x6600 + (q + 8); both halves are handled by one v_pk_add_f16.
  __device__ static inline void accumulate(uint32_t& word, uint32_t p, float rcp, int r) {
    const float a0 = __builtin_amdgcn_fmed3f(mul_f16lo(p, rcp), -8.0f, 7.0f);
    const float a1 = __builtin_amdgcn_fmed3f(mul_f16hi(p, rcp), -8.0f, 7.0f);
    v2h t = __builtin_bit_cast(v2h, pack(a0, a1));
    const v2h magic = {(_Float16)1544.0f, (_Float16)1544.0f};
    t = t + magic;
    word += __builtin_bit_cast(uint32_t, t) << (4 * r);
  }
  static constexpr uint32_t kJunk =
      0x66006600u + (0x66006600u << 4) + (0x66006600u << 8) + (0x66006600u << 12);

  // Packed word of four pairs (nibbles r and r + 4 from pair r), clamping the
  // rounded pair instead of the float32 quotients: rounding is monotonic and
  // -8, 7 are fp16 values, so clamp(rnd(a)) = rnd(clamp(a)). One packed min per
  // pair, plus one packed max when a quotient can round below -8.5 (LOW).
  template <bool LOW>
  __device__ static inline uint32_t word4(const uint32_t (&p)[4], float rcp) {
    const v2h seven = {(_Float16)7.0f, (_Float16)7.0f};
    const v2h minus8 = {(_Float16)-8.0f, (_Float16)-8.0f};
    const v2h magic = {(_Float16)1544.0f, (_Float16)1544.0f};
    uint32_t word = 0u - kJunk;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v2h t = __builtin_bit_cast(v2h, pack(mul_f16lo(p[r], rcp), mul_f16hi(p[r], rcp)));
      t = __builtin_elementwise_min(t, seven);
      if (LOW) t = __builtin_elementwise_max(t, minus8);
      t = t + magic;
      word += __builtin_bit_cast(uint32_t, t) << (4 * r);
    }
    return word;
  }

  // Running extremes of rounded Y pairs, two pairs per step (v_pk_maximum3 /
  // v_pk_minimum3), and max |y| from them as a 16-bit pattern.
  struct Amax {
    v2h hi = {(_Float16)-INFINITY, (_Float16)-INFINITY};
    v2h lo = {(_Float16)INFINITY, (_Float16)INFINITY};
  };
  __device__ static inline void track2(Amax& a, uint32_t p0, uint32_t p1) {
    const v2h y0 = __builtin_bit_cast(v2h, p0), y1 = __builtin_bit_cast(v2h, p1);
    a.hi = __builtin_elementwise_maximum(__builtin_elementwise_maximum(a.hi, y0), y1);
    a.lo = __builtin_elementwise_minimum(__builtin_elementwise_minimum(a.lo, y0), y1);
  }
  __device__ static inline uint32_t amax_bits(const Amax& a) {
    const uint32_t m = pk_absmax16(pk_absmax16(0u, __builtin_bit_cast(uint32_t, a.hi)),
                                   __builtin_bit_cast(uint32_t, a.lo));
    return max(m & 0xFFFFu, m >> 16);
  }
};

template <>
struct FqEpi<BF16T> {
  __device__ static inline uint32_t pack(float a, float b) {
    const v2bf h = {(__bf16)opaque(a), (__bf16)opaque(b)};
    return __builtin_bit_cast(uint32_t, h);
  }
  __device__ static inline uint32_t pack_acc(float a, float b) {
    const v2bf h = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, h);
  }
  __device__ static inline float lo(uint32_t p) { return __builtin_bit_cast(float, p << 16); }
  __device__ static inline float hi(uint32_t p) { return __builtin_bit_cast(float, p & 0xFFFF0000u); }
  // bf16: rounded pair back to float32, then + 12582920 = 1.5 * 2^23 + 8 leaves
  // bits 0x4B400000 + (q + 8). The high element is shifted by 16 + 4r, which
  // drops all of 0x4B400000; the low element's constant part sums to kJunk.
  __device__ static inline void accumulate(uint32_t& word, uint32_t p, float rcp, int r) {
    const float a0 = __builtin_amdgcn_fmed3f(lo(p) * rcp, -8.0f, 7.0f);
    const float a1 = __builtin_amdgcn_fmed3f(hi(p) * rcp, -8.0f, 7.0f);
    const uint32_t t = pack(a0, a1);
    const float f0 = lo(t) + 12582920.0f;
    const float f1 = hi(t) + 12582920.0f;
    word += __builtin_bit_cast(uint32_t, f0) << (4 * r);
    word += __builtin_bit_cast(uint32_t, f1) << (16 + 4 * r);
  }
  static constexpr uint32_t kJunk =
      0x4B400000u + (0x4B400000u << 4) + (0x4B400000u << 8) + (0x4B400000u << 12);

  // Packed word of four pairs (the float32 clamp covers both bounds).
  template <bool LOW>
  __device__ static inline uint32_t word4(const uint32_t (&p)[4], float rcp) {
    uint32_t word = 0u - kJunk;
#pragma unroll
    for (int r = 0; r < 4; ++r) accumulate(word, p[r], rcp, r);
    return word;
  }

  // Code byte B of d from a rounded quotient t (a bf16 value in a float32
  // register, -8.5 <= t < 7.5): one SDWA add of 12582920 = 1.5 * 2^23 + 8,
  // whose float32 sum has a unit ulp, so it rounds t + 8 half to even, which
  // is rint(t) + 8 (8 is even), and leaves that integer (0 .. 15) in the
  // low byte of its bits; dst_sel writes that byte into byte B of d, the
  // other bytes kept (FIRST: cleared). A NaN t (its float32 low half zero)
  // gives byte 0, as v_cvt_pk_u8_f32 of t + 8 does.
  template <int B, bool FIRST>
  __device__ static inline void code_byte(uint32_t& d, float t, float magic) {
    static_assert(!FIRST || B == 0, "the first byte of a word clears the rest");
#define QO_CODE_BYTE(SEL, UNUSED, C)                                                                         \
  asm("v_add_f32_sdwa %0, %1, %2 dst_sel:" SEL " dst_unused:" UNUSED " src0_sel:DWORD src1_sel:DWORD"     \
      : C(d)                                                                                                \
      : "v"(t), "v"(magic))
    if constexpr (FIRST) QO_CODE_BYTE("BYTE_0", "UNUSED_PAD", "=v");
    else if constexpr (B == 1) QO_CODE_BYTE("BYTE_1", "UNUSED_PRESERVE", "+v");
    else if constexpr (B == 2) QO_CODE_BYTE("BYTE_2", "UNUSED_PRESERVE", "+v");
    else QO_CODE_BYTE("BYTE_3", "UNUSED_PRESERVE", "+v");
#undef QO_CODE_BYTE
  }

  // The packed word of four pairs from rounded quotients t[i] (code i):
  // even codes in the bytes of ev, odd codes in the bytes of od, and
  // ev | od << 4 puts code i in nibble i.
  __device__ static inline uint32_t word_from_quotients(const float (&t)[8]) {
    const float magic = 12582920.0f;
    uint32_t ev, od;
    code_byte<0, true>(ev, t[0], magic);
    code_byte<0, true>(od, t[1], magic);
    code_byte<1, false>(ev, t[2], magic);
    code_byte<1, false>(od, t[3], magic);
    code_byte<2, false>(ev, t[4], magic);
    code_byte<2, false>(od, t[5], magic);
    code_byte<3, false>(ev, t[6], magic);
    code_byte<3, false>(od, t[7], magic);
    return ev | (od << 4);
  }

  // The same word as word4 through code bytes: per code the quotient
  // y * rcp clamped to [-8, 7] (v_med3; the clamp commutes with the rounding
  // since -8 and 7 are bf16 values), rounded to bf16 straight into a float32
  // register by one v_cvt_pk_bf16_f32 whose low half is the conversion of 0.0
  // (the bf16 value's float32 bits, low half zero), then code_byte: 10 VALU
  // per pair of codes (the two elements unpacked, two products, two clamps,
  // two conversions, two code bytes).
  __device__ static inline uint32_t word_u8(const uint32_t (&p)[4], float rcp) {
    float t[8];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      // operands are VALU results, never MFMA results
      asm("v_cvt_pk_bf16_f32 %0, 0, %1" : "=v"(t[r]) : "v"(__builtin_amdgcn_fmed3f(lo(p[r]) * rcp, -8.0f, 7.0f)));
      asm("v_cvt_pk_bf16_f32 %0, 0, %1" : "=v"(t[r + 4]) : "v"(__builtin_amdgcn_fmed3f(hi(p[r]) * rcp, -8.0f, 7.0f)));
    }
    return word_from_quotients(t);
  }

  // word_u8 for a token whose largest quotient rounds below 7.5 and whose
  // smallest rounds to -8.5 or above (every code then lies in -8 .. 7 with
  // no clamp; the host picks this form from the clip ratio, kNoClampClip):
  // 8 VALU per pair of codes.
  __device__ static inline uint32_t word_u8_noclamp(const uint32_t (&p)[4], float rcp) {
    float t[8];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      // operands are VALU products, never MFMA results
      asm("v_cvt_pk_bf16_f32 %0, 0, %1" : "=v"(t[r]) : "v"(lo(p[r]) * rcp));
      asm("v_cvt_pk_bf16_f32 %0, 0, %1" : "=v"(t[r + 4]) : "v"(hi(p[r]) * rcp));
    }
    return word_from_quotients(t);
  }

  // max |y| of rounded Y pairs as a 16-bit pattern (sign-cleared bf16 bits
  // order like the values).
  struct Amax {
    uint32_t m = 0u;
  };
  __device__ static inline void track2(Amax& a, uint32_t p0, uint32_t p1) {
    a.m = pk_absmax16(pk_absmax16(a.m, p0), p1);
  }
  __device__ static inline uint32_t amax_bits(const Amax& a) { return max(a.m & 0xFFFFu, a.m >> 16); }
};

// LDS transpose read of 16-bit elements (gfx950 ds_read_b64_tr_b16): within
// each 16-lane group, lane l supplies the address of 4 consecutive elements
// (8-byte aligned), forming row l of a 16 x 4 matrix A; lane i receives
// A[i/4][i%4], A[4 + i/4][i%4], A[8 + i/4][i%4], A[12 + i/4][i%4] — that is,
// A[4e + i/4][i%4] for e = 0..3 (checked on the device).
typedef short v4s16 __attribute__((ext_vector_type(4)));
__device__ inline v4s16 lds_tr16(const void* p) {
  typedef __attribute__((address_space(3))) v4s16* lds_v4s16;
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s16)(__attribute__((address_space(3))) const void*)p);
}
// Two 4-element reads as one 8-element MFMA operand (elements 0..3, 4..7).
template <class V>
__device__ inline V join_tr16(v4s16 lo, v4s16 hi) {
  typedef short v8s16 __attribute__((ext_vector_type(8)));
  const v8s16 w = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  return __builtin_bit_cast(V, w);
}

// Wait until at most N vector-memory operations of this wave are outstanding.
// vmcnt is 6 bits on gfx9 (0..63); the encoding keeps lgkmcnt / expcnt at max.
template <int N>
__device__ inline void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt out of range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

}  // namespace qo
