// The activation rows of the ggml route, quantised: sixteen lanes per run of 256 values in the tile and strip kernels
// (gguf_matvec_q8.hip, gguf_matvec_strips.hip), before they touch a weight; the span, quad, line and block kernels of
// gguf_matvec_q8.hip have lanes of 32 or eight values and take the maxima and the short form from here.
#pragma once

#include <type_traits>

#include "device_common.h"
#include "gguf_q8_math.h"

namespace hyle_hip {
namespace {

typedef short short2v __attribute__((ext_vector_type(2)));

// kCount values of an activation row, sixteen as a rule: neighbours, at any element's address.
template <class TX, int kCount = 16> struct BlockValues {
  static constexpr int kVectors = kCount * Traits<TX>::kSize / 16;
  u32x4 raw[kVectors];
  __device__ __forceinline__ void load(const void *x, size_t first) {
#pragma unroll
    for (int h = 0; h < kVectors; ++h)
      raw[h] = *reinterpret_cast<const u32x4_element *>(static_cast<const char *>(x) + first * Traits<TX>::kSize + 16 * h);
  }
  __device__ __forceinline__ void values(float (&v)[kCount]) const {
#pragma unroll
    for (int h = 0; h < kVectors; ++h) {
      float piece[Traits<TX>::kVec];
      Traits<TX>::unpack(raw[h], piece);
#pragma unroll
      for (int e = 0; e < Traits<TX>::kVec; ++e) v[Traits<TX>::kVec * h + e] = piece[e];
    }
  }
  // f32 bits of the largest value that is not negative and of the largest magnitude among the others, 0 where
  // there is none.  Compared as stored: bit patterns of one sign are in the order of their magnitudes, NaN last.
  __device__ __forceinline__ void extremes(uint32_t &positive, uint32_t &negative) const {
    if constexpr (Traits<TX>::kSize == 4) {
      int above = (int)raw[0].x;
      uint32_t below = raw[0].x;
#pragma unroll
      for (int i = 1; i < kCount; ++i) {
        above = max(above, (int)raw[i / 4][i % 4]);
        below = max(below, raw[i / 4][i % 4]);
      }
      positive = above < 0 ? 0u : (uint32_t)above;
      negative = (int)below < 0 ? below & 0x7FFFFFFFu : 0u;
    } else {
      typedef short i16x2 __attribute__((ext_vector_type(2)));
      typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
      i16x2 above = __builtin_bit_cast(i16x2, (uint32_t)raw[0].x);
      u16x2 below = __builtin_bit_cast(u16x2, (uint32_t)raw[0].x);
#pragma unroll
      for (int i = 1; i < kCount / 2; ++i) {
        above = __builtin_elementwise_max(above, __builtin_bit_cast(i16x2, (uint32_t)raw[i / 4][i % 4]));
        below = __builtin_elementwise_max(below, __builtin_bit_cast(u16x2, (uint32_t)raw[i / 4][i % 4]));
      }
      const int high = max((int)above.x, (int)above.y);
      const uint32_t low = max((uint32_t)below.x, (uint32_t)below.y);
      positive = f32_bits(widened((uint32_t)max(high, 0)));
      negative = f32_bits(widened((low & 0x8000u) != 0 ? low & 0x7FFFu : 0u));
    }
  }
  static __device__ __forceinline__ float widened(uint32_t half) {
    if constexpr (std::is_same_v<TX, BF16>) return bits_f32(half << 16);
    else return f16_to_f32((uint16_t)half);
  }
};

// The largest over 1, 2, 4, 8, 16 or 32 neighbouring lanes.
template <int kLanes> __device__ __forceinline__ uint32_t lanes_max(uint32_t v) {
  if constexpr (kLanes > 1) v = max(v, (uint32_t)dpp_move<kDppSwap1>((int)v));
  if constexpr (kLanes > 2) v = max(v, (uint32_t)dpp_move<kDppSwap2>((int)v));
  if constexpr (kLanes > 4) v = max(v, (uint32_t)dpp_move<kDppHalfMirror>((int)v));
  if constexpr (kLanes > 8) v = max(v, (uint32_t)dpp_move<kDppRowMirror>((int)v));
  if constexpr (kLanes > 16) v = max(v, (uint32_t)__shfl_xor((int)v, 16, kWaveLanes));
  return v;
}

// 127 / b correctly rounded for b from 2^-60 to 2^61: the hardware's reciprocal, a Newton step and a correction of
// the quotient by its exact remainder, right for every mantissa of b with a reciprocal up to one unit off.  It is
// six instructions where the full division, which scales its operands, is eleven.  (1 / b is not to be had this way
// without knowing the reciprocal of a mantissa of all ones: from an estimate that is off the steps end one unit short.)
__device__ __forceinline__ float quotient_of_127(float b) {
  const float rough = __builtin_amdgcn_rcpf(b);
  const float inverse = __builtin_fmaf(__builtin_fmaf(-b, rough, 1.0f), rough, rough);
  const float q = 127.0f * inverse;
  return __builtin_fmaf(__builtin_fmaf(-b, q, 127.0f), inverse, q);
}
// b / 127 the same way
__device__ __forceinline__ float over_127(float b) {
  constexpr float kInverse = 1.0f / 127.0f;
  const float q = b * kInverse;
  return __builtin_fmaf(__builtin_fmaf(-127.0f, q, b), kInverse, q);
}

// What the short form below needs to know of a block that kLanes neighbouring lanes share, kCount values each: f32 bits of
// its largest magnitude, of its largest value that is not negative and of its largest magnitude among the others
// (Q8_0, kSmall: all three the first, NaN if there is one).
struct BlockTop {
  uint32_t bits, positive, negative;
  bool small;
  // largest magnitude between 2^-60 and 2^61 and (Q8_K, where its sign counts) not met with both signs
  __device__ __forceinline__ bool regular() const { return bits >= (67u << 23) && bits < (188u << 23) && (small || positive != negative); }
};
template <bool kSmall, int kLanes, class TX, int kCount>
__device__ __forceinline__ BlockTop block_top(const BlockValues<TX, kCount> &fetched, const float (&v)[kCount]) {
  BlockTop top;
  top.small = kSmall;
  if constexpr (kSmall) {
    float largest = 0.0f;
#pragma unroll
    for (int e = 0; e < kCount; e += 2)
      largest = __builtin_elementwise_maximum(__builtin_elementwise_maximum(__builtin_fabsf(v[e]), __builtin_fabsf(v[e + 1])), largest);
    top.positive = top.negative = top.bits = lanes_max<kLanes>(f32_bits(largest) & 0x7FFFFFFFu);
  } else {
    fetched.extremes(top.positive, top.negative);
    top.positive = lanes_max<kLanes>(top.positive), top.negative = lanes_max<kLanes>(top.negative);
    top.bits = max(top.positive, top.negative);
  }
  return top;
}
// The short form, for regular blocks: a code is the low byte of value * factor + 1.5 * 2^23, rounded to the nearest
// integer, ties to even, and no more than 127 in magnitude.
template <bool kSmall> __device__ __forceinline__ void short_factors(const BlockTop &top, float &factor, float &stored) {
  factor = quotient_of_127(bits_f32(top.bits));
  if constexpr (kSmall) {
    stored = f16_to_f32(f32_to_f16(over_127(bits_f32(top.bits))));
  } else {
    factor = top.positive > top.negative ? -factor : factor;
    stored = 1.0f / factor;
  }
}
__device__ __forceinline__ uint32_t short_codes(float v0, float v1, float v2, float v3, float factor) {
  const uint32_t code[4] = {f32_bits(v0 * factor + 12582912.0f), f32_bits(v1 * factor + 12582912.0f), f32_bits(v2 * factor + 12582912.0f),
                            f32_bits(v3 * factor + 12582912.0f)};
  return __builtin_amdgcn_perm(__builtin_amdgcn_perm(code[3], code[2], 0x0C0C0400u), __builtin_amdgcn_perm(code[1], code[0], 0x0C0C0400u), 0x05040100u);
}

// Sixteen lanes quantise a run of 256 values of an activation row, sixteen values per lane u: one Q8_K block, or eight
// Q8_0 blocks of two lanes each.  Regular blocks take the short form; any other (zeros, NaN, infinities) sends the wave the
// long way.
template <int kKind, class TX>
__device__ __forceinline__ void quantise_block(const BlockValues<TX> &fetched, uint32_t lane, unsigned char *codes, float *scale, uint32_t scale_step,
                                               int *sums, uint32_t sum_step) {
  constexpr bool kSmall = kKind >= 2;  // blocks of 32
  constexpr int kLanes = kSmall ? 2 : 16;
  const uint32_t u = lane % 16;
  float v[16];
  fetched.values(v);
  const BlockTop block = block_top<kSmall, kLanes>(fetched, v);
  float factor = 0.0f, stored = 0.0f;
  uint32_t words[4];
  if (__builtin_expect(__ballot(!block.regular()) == 0, 1)) {
    short_factors<kSmall>(block, factor, stored);
#pragma unroll
    for (int w = 0; w < 4; ++w) words[w] = short_codes(v[4 * w], v[4 * w + 1], v[4 * w + 2], v[4 * w + 3], factor);
  } else {
    float largest = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) largest = __builtin_fmaxf(largest, __builtin_fabsf(v[e]));  // a NaN is no candidate
    const float top = bits_f32(lanes_max<kLanes>(f32_bits(largest)));
    if constexpr (kSmall) {
      if (top != 0.0f) {
        stored = f16_to_f32(f32_to_f16(top / 127.0f));
        factor = 127.0f / top;
      }
    } else {
      // the sign of the block's first value of that magnitude: of the lowest lane that has one
      bool below_zero = false;
#pragma unroll
      for (int e = 15; e >= 0; --e) below_zero = __builtin_fabsf(v[e]) == top ? v[e] < 0.0f : below_zero;
      const uint64_t has = __ballot(largest == top), below = __ballot(below_zero);
      const uint32_t own_has = (uint32_t)(has >> (lane & 48u)) & 0xFFFFu, own_below = (uint32_t)(below >> (lane & 48u));
      if (top != 0.0f) {
        const float value = (own_below >> __builtin_ctz(own_has)) & 1u ? -top : top;
        factor = -127.0f / value;
        stored = 1.0f / factor;
      }
    }
    // nearest integer, ties to even, at most 127 (a block of zeros: factor 0); only the low bytes are kept
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      int code[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) code[e] = (int)__builtin_rintf(v[4 * w + e] * factor);
      const short2v most = {127, 127};
      const short2v low = __builtin_elementwise_min(__builtin_bit_cast(short2v, __builtin_amdgcn_cvt_pk_i16(code[0], code[1])), most);
      const short2v high = __builtin_elementwise_min(__builtin_bit_cast(short2v, __builtin_amdgcn_cvt_pk_i16(code[2], code[3])), most);
      words[w] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, high), __builtin_bit_cast(uint32_t, low), 0x06040200u);
    }
  }
  const u32x4 whole = {words[0], words[1], words[2], words[3]};
  // Q8_0 in place: 48 bytes per block, its codes where its quants lie in the 48 bytes from its first vector
  if constexpr (kKind >= 3) *reinterpret_cast<u32x4_element *>(codes + 50 * (u / 2) + 2 + 16 * (u % 2)) = whole;
  else reinterpret_cast<u32x4 *>(codes)[u] = whole;
  if constexpr (kKind == 0) {
    int sum = dot4(0x01010101u, words[0], dot4(0x01010101u, words[1], dot4(0x01010101u, words[2], dot4(0x01010101u, words[3], 0))));
    sum += dpp_move<kDppSwap1>(sum);  // the two lanes of a sub-block
    if (u % 2 == 0) sums[(u / 2) * sum_step] = sum;
  }
  if constexpr (kSmall) {
    if (u % 2 == 0) scale[(u / 2) * scale_step] = stored;
  } else {
    if (u == 0) *scale = stored;
  }
}

}  // namespace
}  // namespace hyle_hip
