// Register dequantization of packed weights into MFMA operand words, shared by the MFMA
// GEMM (qgemm_tile_kernel.h) and the dequant entry point (qgemm_pack.hip), so the values the
// GEMM multiplies are exactly the ones mlxr_qgemm_dequant returns.
//
// A "word" is 8 consecutive weights of a 32-weight sub-block (word kk = weights 8kk ..
// 8kk+7) as four packed pairs of the MFMA element type (bf16, or fp16 for fp16
// activations).  Each value is the exact GGUF fp32 weight, rounded to nearest even:
//   Q4_K  fma(d*sc, q, -(dmin*m))       (d*sc, q*d*sc and dmin*m exact; one rounding)
//   Q5_K  as Q4_K with q in 0..31
//   Q6_K  (d*sc) * (q - 32)             (exact; q - 32 formed exactly in fp32)
//   Q8_0  d * q                         (exact)
//   Q4_0  (q - 8) * d                   (exact)
//   Q4_1  fma(q, d, m)                  (q*d exact; one rounding)
// (the products keep the sign of zero of the GGUF formulas, which an fma with an
// offset term would not: fma(a, 32, -32a) is +0 for negative a).  The GEMM kernels take
// the MM variant: for Q6_K, Q8_0 and Q4_0 it forms the same values with one fma
// (fma(a, q, -c*a) rounds a*q - c*a, which is exactly a*(q - c), once), one operation per
// weight fewer; only an exact zero may differ in sign, which no product sum can see.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qgemm_device.h"
#include "qgemm_internal.h"

namespace mlxr {

typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2_t;

enum XType : int { X_BF16 = 0, X_F16 = 1 };

// Two floats -> packed pair of the MFMA element type, round to nearest even.
template <int XT>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  if constexpr (XT == X_BF16) {
    return pack_bf16x2(lo, hi);
  } else {
    const f32x2_t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
  }
}

// An empty asm that makes later uses of v depend on this point in the program (used to
// order work against explicit waits and inside the MFMA stream).
template <typename T>
__device__ __forceinline__ void pin(T& v) {
  asm volatile("" : "+v"(v));
}

template <int QT>
struct Raw;
template <>
struct Raw<QT_Q4_K> {
  u32x4_t q;
  __device__ void pin_all() { pin(q); }
};
template <>
struct Raw<QT_Q6_K> {
  u32x4_t ql;
  u32x2_t qh;
  __device__ void pin_all() {
    pin(ql);
    pin(qh);
  }
};
template <>
struct Raw<QT_Q8_0> {
  u32x4_t a, b;
  uint32_t d;
  __device__ void pin_all() {
    pin(a);
    pin(b);
    pin(d);
  }
};

// Q5_K: the Q4_K nibbles plus the sub-block's fifth bits (q5h_bit order).
template <>
struct Raw<QT_Q5_K> {
  u32x4_t q;
  uint32_t qh;
  __device__ void pin_all() {
    pin(q);
    pin(qh);
  }
};

// Q4_0 / Q4_1: one 32-weight block (4 pair-interleaved words) and its scale word
// (fp16 d, plus fp16 m in the high half for Q4_1).
template <>
struct Raw<QT_Q4_0> {
  u32x4_t q;
  uint32_t d;
  __device__ void pin_all() {
    pin(q);
    pin(d);
  }
};
template <>
struct Raw<QT_Q4_1> {
  u32x4_t q;
  uint32_t d;
  __device__ void pin_all() {
    pin(q);
    pin(d);
  }
};

// Header bytes of one super-block as loaded; decoded once per four steps.
template <int QT>
struct Hdr {
  u32x4_t h;   // Q4_K: 8 x u16 lane-sliced entries; Q6_K: 16 int8 scales
  uint32_t d;  // Q6_K: fp16 d
  __device__ void pin_all() {
    pin(h);
    if constexpr (QT == QT_Q6_K) pin(d);
  }
};
// Decoded per-sub-block factors for the four sub-blocks (h, h+2, h+4, h+6) a lane owns
// in the current super-block.  Scales of values are kept times SUB24 (see half_scale).
template <int QT>
struct Scales {
  float a[4], b[4];  // Q4_K: d*sc * 2^24, -(dmin*m).  Q6_K: d*sc * 2^24 of the two 16-weight groups.
};

// The weight codes reach fp32 as subnormal halves: a code masked into bits 0..9 of a 16-bit
// half is the fp16 number code * 2^-24 (code * 2^-20 when it sits four bits up), and
// v_fma_mix_f32 multiplies a half of a register by an fp32 factor and adds in one rounding,
// so fma(a * 2^24, half, c) is exactly fma(a, code, c).  Against converting each byte with
// v_cvt_f32_ubyteN and then multiplying, that is one instruction per weight fewer of those
// that issue at half rate (conversions, mix and packed conversions alike: 1.8 ns per
// wavefront instruction and SIMD on MI355X, where mask and shift take 0.95 ns): eight Q4_K
// weights take 29 ns instead of 35 ns with four wavefronts on a SIMD, 31 instead of 39 ns
// with two, 39 instead of 52 ns with one.
constexpr float SUB24 = 16777216.f;
typedef __attribute__((ext_vector_type(2))) _Float16 half2_t;

template <int QT>
__device__ __forceinline__ void decode_hdr(const Hdr<QT>& h, int half, Scales<QT>& s) {
  if constexpr (QT == QT_Q4_K || QT == QT_Q5_K) {
    const uint32_t dd = q4k_dd(make_uint4(h.h[0], h.h[1], h.h[2], h.h[3]));
    const float d = f16_bits_to_f32(dd & 0xffffu) * SUB24, dmin = f16_bits_to_f32(dd >> 16);
    const uint32_t w[4] = {h.h[0], h.h[1], h.h[2], h.h[3]};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      // entry j = 2q + half sits in word q, half `half`
      const uint32_t f = (half ? (w[q] >> 16) : w[q]) & 0xfffu;
      s.a[q] = d * (float)(f & 63u);
      s.b[q] = -(dmin * (float)(f >> 6));
    }
  } else if constexpr (QT == QT_Q6_K) {
    const float d = f16_bits_to_f32(h.d & 0xffffu) * SUB24;
    const uint32_t w[4] = {h.h[0], h.h[1], h.h[2], h.h[3]};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      // sub-block j = 2q + half uses scales 2j, 2j + 1: bytes 4q + 2half, +1 = word q
      const uint32_t v = half ? (w[q] >> 16) : w[q];
      s.a[q] = d * (float)(int8_t)(v & 0xffu);
      s.b[q] = d * (float)(int8_t)((v >> 8) & 0xffu);
    }
  }
}

// Word kk of a sub-block is computed as a prelude and four quarter tasks (one packed
// pair each: weights (0,1), (2,3), (4,5), (6,7) of the word), so the GEMM can spread the
// work one task per MFMA.  q selects the sub-block's scales (sub-block 2q + half of the
// super-block, see decode_hdr).
template <int QT>
struct WordTmp {
  uint32_t w, l, x, z;  // the word's nibbles, those of its bytes 1 and 3 moved down, high bits (Q8_0: codes)
  float a, a4, c;    // scale of a code at bit 0 of its half, at bit 4; the added term
};

template <int QT, int kk, bool MM = false>
__device__ __forceinline__ void word_prelude(const Raw<QT>& r, const Scales<QT>& s, int q, WordTmp<QT>& t) {
  if constexpr (QT == QT_Q8_0) {
    // int8 q -> q + 128; halves of w: weights 0, 2 of the first int8 word, of l: 1, 3; x and z
    // the second word's.  (Pinned: else the compiler takes them apart again into one extract
    // per weight.)
    uint32_t w0 = kk < 2 ? r.a[2 * kk] : r.b[2 * kk - 4];
    uint32_t w1 = kk < 2 ? r.a[2 * kk + 1] : r.b[2 * kk - 3];
    pin(w0);
    pin(w1);
    t.w = (w0 ^ 0x00800080u) & 0x00FF00FFu;
    t.l = ((w0 >> 8) ^ 0x00800080u) & 0x00FF00FFu;
    t.x = (w1 ^ 0x00800080u) & 0x00FF00FFu;
    t.z = ((w1 >> 8) ^ 0x00800080u) & 0x00FF00FFu;
    pin(t.w);
    pin(t.l);
    pin(t.x);
    pin(t.z);
    const float d = f16_bits_to_f32(r.d & 0xffffu);
    t.a = d * SUB24;
    t.c = MM ? -128.f * d : -128.f;
    return;
  } else if constexpr (QT == QT_Q6_K) {
    t.w = r.ql[kk];
    t.x = (kk & 1) ? (r.qh[kk >> 1] >> 8) : r.qh[kk >> 1];
    t.a = (kk < 2) ? s.a[q] : s.b[q];
    t.c = MM ? t.a * (-32.f / SUB24) : -32.f;
  } else {
    t.w = r.q[kk];
    if constexpr (QT == QT_Q4_0 || QT == QT_Q4_1) {
      const float d = f16_bits_to_f32(r.d & 0xffffu);
      t.a = d * SUB24;
      t.c = QT == QT_Q4_0 ? (MM ? -8.f * d : -8.f) : f16_bits_to_f32(r.d >> 16);
    } else {
      if constexpr (QT == QT_Q5_K) t.x = r.qh;
      t.a = s.a[q];
      t.c = s.b[q];
    }
  }
  pin(t.w);
  t.l = t.w >> 8;
  t.a4 = t.a * 0.0625f;
}

// v shifted so that bit `from` comes to bit `at`.
template <int from, int at>
__device__ __forceinline__ uint32_t move_bits(uint32_t v) {
  if constexpr (at >= from) return v << (at - from);
  else return v >> (from - at);
}

// The codes of pair qq of word kk as subnormal halves.  Pairs 0 and 2 take the low nibbles
// of their bytes (bits 0 and 16), pairs 1 and 3 the high ones in place (bits 4 and 20), with
// their high bits on top.
template <int QT, int kk, int qq>
__device__ __forceinline__ uint32_t pair_codes(const WordTmp<QT>& t) {
  const uint32_t n = ((qq & 2) ? t.l : t.w) & ((qq & 1) ? 0x00F000F0u : 0x000F000Fu);
  if constexpr (QT == QT_Q5_K) {
    // the fifth bits of word kk's pairs sit at bits 2kk, 2kk + 1, 2kk + 8, 2kk + 9 of each half
    constexpr int from = 2 * kk + (qq & 1) + 4 * (qq & 2), at = (qq & 1) ? 8 : 4;
    const uint32_t h = move_bits<from, at>(t.x);
    return n | (h & ((qq & 1) ? 0x01000100u : 0x00100010u));
  } else if constexpr (QT == QT_Q6_K) {
    // the two high bits of pair qq sit at bits 2qq, 2qq + 1 of each half
    constexpr int from = 2 * qq, at = (qq & 1) ? 8 : 4;
    const uint32_t h = move_bits<from, at>(t.x);
    return n | (h & ((qq & 1) ? 0x03000300u : 0x00300030u));
  } else {
    return n;
  }
}

// One weight: half hi of the codes v, a the scale of a code at their position.
template <int QT, bool MM>
__device__ __forceinline__ float word_value(uint32_t v, int hi, float a, float c, bool at4) {
  const half2_t hv = __builtin_bit_cast(half2_t, v);
  if constexpr (MM || QT == QT_Q4_K || QT == QT_Q5_K || QT == QT_Q4_1) return __builtin_fmaf(a, (float)hv[hi], c);
  // the product form of the formulas: (code + c) exactly, then times the scale
  return __builtin_fmaf(at4 ? SUB24 / 16.f : SUB24, (float)hv[hi], c) * (a * ((at4 ? 16.f : 1.f) / SUB24));
}

template <int QT, int XT, int kk, int qq, bool MM = false>
__device__ __forceinline__ uint32_t word_quarter(const WordTmp<QT>& t) {
  if constexpr (QT == QT_Q8_0) {
    return pack2<XT>(word_value<QT, MM>((qq & 2) ? t.x : t.w, qq & 1, t.a, t.c, false),
                     word_value<QT, MM>((qq & 2) ? t.z : t.l, qq & 1, t.a, t.c, false));
  } else {
    const uint32_t v = pair_codes<QT, kk, qq>(t);
    const float a = (qq & 1) ? t.a4 : t.a;
    return pack2<XT>(word_value<QT, MM>(v, 0, a, t.c, qq & 1), word_value<QT, MM>(v, 1, a, t.c, qq & 1));
  }
}

// The whole word (dequant entry point; MM: GEMM kernels).
template <int QT, int XT, int kk, bool MM = false>
__device__ __forceinline__ uint4 dequant_word(const Raw<QT>& r, const Scales<QT>& s, int q) {
  WordTmp<QT> t;
  word_prelude<QT, kk, MM>(r, s, q, t);
  return make_uint4(word_quarter<QT, XT, kk, 0, MM>(t), word_quarter<QT, XT, kk, 1, MM>(t),
                    word_quarter<QT, XT, kk, 2, MM>(t), word_quarter<QT, XT, kk, 3, MM>(t));
}

// Plain (compiler-visible) loads of sub-block sb of row n and of its super-block header,
// for the dequant entry point.
template <int QT>
__device__ __forceinline__ void load_sub_plain(const PlanePtrs& P, int K, int n, int sb, Raw<QT>& r, Hdr<QT>& h) {
  const size_t nsub = (size_t)(K >> 5), nsb = (size_t)(K >> 8);
  const size_t s = (size_t)n * nsub + (size_t)sb;
  const size_t g = (size_t)n * nsb + (size_t)(sb >> 3);
  if constexpr (QT == QT_Q4_K) {
    r.q = *(const u32x4_t*)(P.p[0] + s * 16);
    h.h = *(const u32x4_t*)(P.p[1] + g * 16);
  } else if constexpr (QT == QT_Q5_K) {
    r.q = *(const u32x4_t*)(P.p[0] + s * 16);
    r.qh = *(const uint32_t*)(P.p[1] + s * 4);
    h.h = *(const u32x4_t*)(P.p[2] + g * 16);
  } else if constexpr (QT == QT_Q4_0) {
    r.q = *(const u32x4_t*)(P.p[0] + s * 16);
    r.d = *(const uint16_t*)(P.p[1] + s * 2);
  } else if constexpr (QT == QT_Q4_1) {
    r.q = *(const u32x4_t*)(P.p[0] + s * 16);
    r.d = *(const uint32_t*)(P.p[1] + s * 4);
  } else if constexpr (QT == QT_Q6_K) {
    r.ql = *(const u32x4_t*)(P.p[0] + s * 16);
    r.qh = *(const u32x2_t*)(P.p[1] + s * 8);
    h.h = *(const u32x4_t*)(P.p[2] + g * 16);
    h.d = *(const uint16_t*)(P.p[3] + g * 2);
  } else {
    r.a = *(const u32x4_t*)(P.p[0] + s * 32);
    r.b = *(const u32x4_t*)(P.p[0] + s * 32 + 16);
    r.d = *(const uint16_t*)(P.p[1] + s * 2);
  }
}

// The 32 weights of sub-block sb of row n as four words of element type XT.
template <int QT, int XT>
__device__ __forceinline__ void dequant_sub_words(const PlanePtrs& P, int K, int n, int sb, uint4* out) {
  Raw<QT> r;
  Hdr<QT> h;
  load_sub_plain<QT>(P, K, n, sb, r, h);
  Scales<QT> sc;
  decode_hdr<QT>(h, sb & 1, sc);
  const int q = (sb & 7) >> 1;
  out[0] = dequant_word<QT, XT, 0>(r, sc, q);
  out[1] = dequant_word<QT, XT, 1>(r, sc, q);
  out[2] = dequant_word<QT, XT, 2>(r, sc, q);
  out[3] = dequant_word<QT, XT, 3>(r, sc, q);
}

}  // namespace mlxr
