// The activation split's arithmetic: BF16 values of one 128-column block as s
// (hi + lo / 16) with hi and lo E4M3 and s a power of two.
#pragma once

#include "common.h"

namespace glm53 {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef short i16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

// Hardware E4M3 conversion (round to nearest even) of a pair of BF16 values
// over the scale s, both |x / s| <= 448, into bytes 0-1 (kUpper false) or 2-3
// of hi_word, and of their residuals 16 (x / s - hi) into the same bytes of
// lo_word; the other bytes are kept.  The scaled conversions divide by a
// power of two as they convert: their codes equal those of the conversions
// of x / s and 16 (x / s - hi) for every BF16 x (tests/test_gpu_split.py, both
// ends of the scales they serve included), seven instructions a pair instead
// of twelve.
template <bool kUpper>
__device__ __forceinline__ void encode_pair_e4m3(uint32_t x, float s, uint32_t& hi_word, uint32_t& lo_word) {
  hi_word = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(
                                             __builtin_bit_cast(i16x2_t, hi_word), __builtin_bit_cast(bf16x2_t, x), s,
                                             kUpper));
  const f32x2_t h = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hi_word, s, kUpper);  // hi s
  const float r0 = __uint_as_float(x << 16) - h[0], r1 = __uint_as_float(x & 0xFFFF0000u) - h[1];
  lo_word = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(
                                             __builtin_bit_cast(i16x2_t, lo_word), r0, r1, s * 0.0625f, kUpper));
}

// V consecutive BF16 values as raw words: V = 8 is one 16-byte load (the
// pointer 16-byte aligned), V = 1 or 2 are 2-byte loads.
template <int V>
struct Bf16Run {
  uint32_t w[(V + 1) / 2];
  __device__ __forceinline__ void load(const uint16_t* p) {
    if constexpr (V == 8) {
      const uint4 r = *reinterpret_cast<const uint4*>(p);
      w[0] = r.x, w[1] = r.y, w[2] = r.z, w[3] = r.w;
    } else {
#pragma unroll
      for (int i = 0; i < (V + 1) / 2; ++i) w[i] = 0u;
#pragma unroll
      for (int i = 0; i < V; ++i) w[i >> 1] |= static_cast<uint32_t>(p[i]) << (16 * (i & 1));
    }
  }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < (V + 1) / 2; ++i) w[i] = 0u;
  }
  __device__ __forceinline__ float get(int i) const {
    return __uint_as_float(i & 1 ? (w[i >> 1] & 0xffff0000u) : (w[i >> 1] << 16));
  }
};

// The largest |x| over a DPP row's 16 lanes, in each of them.
__device__ __forceinline__ float row16_amax(float v) {
  v = fmaxf(v, dpp_f32<0xB1>(v));     // quad_perm [1,0,3,2]
  v = fmaxf(v, dpp_f32<0x4E>(v));     // quad_perm [2,3,0,1]
  v = fmaxf(v, dpp_f32<0x141>(v));    // row_half_mirror
  return fmaxf(v, dpp_f32<0x140>(v));  // row_mirror
}

// The largest |x| of a lane's values, NaNs left out; has_nan: there are some.
// On the BF16 bits, two values per instruction.
template <int V>
__device__ __forceinline__ uint32_t lane_amax_bits(const Bf16Run<V>& x) {  // NaNs included
  uint32_t m = 0;
#pragma unroll
  for (int i = 0; i < (V + 1) / 2; ++i) m = max_u16x2(m, x.w[i] & 0x7FFF7FFFu);
  return max(m & 0xFFFFu, m >> 16);
}
template <int V>
__device__ __forceinline__ float lane_amax(const Bf16Run<V>& x, bool& has_nan) {
  const uint32_t u = lane_amax_bits<V>(x);
  has_nan = u > 0x7F80u;
  float amax = __uint_as_float(u << 16);
  if (has_nan) {
    amax = 0.0f;
#pragma unroll
    for (int i = 0; i < V; ++i) amax = fmaxf(amax, fabsf(x.get(i)));
  }
  return amax;
}

// A block's scale s = 2^ceil(log2(amax / 448)), so that amax / s lies in (224,
// 448], and 1 / s; both 1 for an all-zero or non-finite block.  448 = 1.75
// 2^8: the exponent is amax's less 8, plus one where its significand is over
// 1.75, and not below -126.
struct SplitScale {
  float s, inv;
  bool plain;  // a finite block, and 2^-95 <= s <= 2^119: neither s / 16 nor 448 s leaves the normal range
};
__device__ __forceinline__ SplitScale split_scale(float amax) {
  const uint32_t u = __float_as_uint(amax);
  int code = static_cast<int>(u >> 23) + ((u & 0x7FFFFFu) > 0x600000u ? 1 : 0) - 8;
  code = max(code, 1);
  if (u == 0u || u >= 0x7F800000u) code = 127;
  return {__uint_as_float(static_cast<uint32_t>(code) << 23), __uint_as_float(static_cast<uint32_t>(254 - code) << 23),
          u < 0x7F800000u && code >= 32 && code <= 246};
}

template <int V>
struct SplitHalf {
  static constexpr int value = V;
};

// V values of a block of scale s (s.plain, no NaN in the lane) as hi and lo
// codes packed four to a word: every |x / s| <= 448, the range of E4M3; the
// residual |x / s - hi| <= 16 makes 16 times it lie within +-256.
template <int V>
__device__ __forceinline__ void split_encode_plain(const Bf16Run<V>& x, const SplitScale& s,
                                                   uint32_t (&hi)[(V + 3) / 4], uint32_t (&lo)[(V + 3) / 4]) {
#pragma unroll
  for (int w = 0; w < (V + 3) / 4; ++w) {
    hi[w] = lo[w] = 0;
    encode_pair_e4m3<false>(x.w[2 * w], s.s, hi[w], lo[w]);
    if constexpr (V >= 4) encode_pair_e4m3<true>(x.w[2 * w + 1], s.s, hi[w], lo[w]);
  }
}

// The same for any values: x / s saturates at +-448 (NaN too, under its
// sign), then the unscaled conversions, exact encodings up to there; the same
// codes where both forms apply.
template <int V>
__device__ __forceinline__ void split_encode_any(const Bf16Run<V>& x, const SplitScale& s,
                                                 uint32_t (&hi)[(V + 3) / 4], uint32_t (&lo)[(V + 3) / 4]) {
  auto sat = [](float v) { return __builtin_copysignf(fminf(fabsf(v), 448.0f), v); };
  auto pair = [&](uint32_t xw, uint32_t& h, uint32_t& l, auto upper) {
    const float q0 = __uint_as_float(xw << 16) * s.inv, q1 = __uint_as_float(xw & 0xFFFF0000u) * s.inv;
    h = static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(sat(q0), sat(q1), static_cast<int>(h), upper.value));
    const float r0 = (q0 - __builtin_amdgcn_cvt_f32_fp8(static_cast<int>(h), 2 * upper.value)) * 16.0f;
    const float r1 = (q1 - __builtin_amdgcn_cvt_f32_fp8(static_cast<int>(h), 2 * upper.value + 1)) * 16.0f;
    l = static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(sat(r0), sat(r1), static_cast<int>(l), upper.value));
  };
#pragma unroll
  for (int w = 0; w < (V + 3) / 4; ++w) {
    hi[w] = lo[w] = 0;
    pair(x.w[2 * w], hi[w], lo[w], SplitHalf<0>{});
    if constexpr (V >= 4) pair(x.w[2 * w + 1], hi[w], lo[w], SplitHalf<1>{});
  }
}

// Either form for the whole wavefront, so that the unusual one's instructions
// lie out of the way; has_nan: the lane's values hold a NaN.
template <int V>
__device__ __forceinline__ void split_encode(const Bf16Run<V>& x, const SplitScale& s, bool has_nan,
                                             uint32_t (&hi)[(V + 3) / 4], uint32_t (&lo)[(V + 3) / 4]) {
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(!s.plain || has_nan) == 0, 1)) split_encode_plain<V>(x, s, hi, lo);
  else split_encode_any<V>(x, s, hi, lo);
}

}  // namespace glm53
