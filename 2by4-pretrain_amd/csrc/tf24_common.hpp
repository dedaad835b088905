// Shared device/host helpers for the gfx950 2:4 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <initializer_list>
#include <type_traits>

#include "tf24.h"

namespace tf24 {

// ---------------------------------------------------------------- error reporting (host)
void set_error(const char* fmt, ...);
int fail(int code, const char* fmt, ...);
int check_launch(const char* what);
// TF24_ERR_STRIDE unless every listed pointer (NULL is skipped) is aligned to `bytes`: the kernels
// use 128-bit (metadata and byte masks: 64-bit) accesses and do not handle split lines
int check_aligned(const char* fn, int bytes, std::initializer_list<const void*> ptrs);

// ---------------------------------------------------------------- element types
struct f16_t { uint16_t bits; };
struct bf16_t { uint16_t bits; };
struct e4m3_t { uint8_t bits; };
struct e5m2_t { uint8_t bits; };
struct i8_t { uint8_t bits; };      // two's-complement int8

template <typename T> struct dtype_of;
template <> struct dtype_of<float> { static constexpr int value = TF24_F32; };
template <> struct dtype_of<f16_t> { static constexpr int value = TF24_F16; };
template <> struct dtype_of<bf16_t> { static constexpr int value = TF24_BF16; };
template <> struct dtype_of<e4m3_t> { static constexpr int value = TF24_E4M3; };
template <> struct dtype_of<e5m2_t> { static constexpr int value = TF24_E5M2; };
template <> struct dtype_of<i8_t> { static constexpr int value = TF24_I8; };
template <> struct dtype_of<int32_t> { static constexpr int value = TF24_I32; };
__host__ __device__ inline bool is_float8(int dt) { return dt == TF24_E4M3 || dt == TF24_E5M2; }
// value types stored one byte per element: 128 dense columns per panel, int32 metadata words
__host__ __device__ inline bool is_8bit(int dt) { return is_float8(dt) || dt == TF24_I8; }
template <> struct dtype_of<uint8_t> { static constexpr int value = TF24_U8; };

// Panel form of the metadata, [k/32][m][4 bytes]: byte offset of metadata byte `mbyte` (= dense column / 8)
// of row `row` of a matrix with m rows.
__host__ __device__ inline int64_t panel_meta_offset(int64_t mbyte, int64_t row, int64_t m) {
  return ((mbyte >> 2) * m + row) * 4 + (mbyte & 3);
}

// CUTLASS form of the metadata (reorder_meta + ColumnMajorInterleaved<2>, reference csrc .cu:826-851):
// byte offset of metadata byte `mbyte` of row `row`.  WB = bytes per metadata word (2: int16 words of
// 16-bit values, 4: int32 words of 8-bit values).  Word (row, c) moves to row
// row/G*G + (row%8)*I + (row%G)/8 with (G, I) = (32, 4) | (16, 2), is swapped inside 2 x 2 blocks (even
// row, odd column <-> odd row, even column) and lands at word (c'/2)*2m + 2*row' + c'%2.
template <int WB>
__host__ __device__ inline int64_t cutlass_meta_offset(int64_t mbyte, int64_t row, int64_t m) {
  constexpr int G = WB == 2 ? 32 : 16, I = WB == 2 ? 4 : 2;
  const int64_t c = mbyte / WB;
  int64_t dr = row / G * G + (row % 8) * I + (row % G) / 8, dc = c;
  if ((dr & 1) == 0 && (dc & 1) == 1) { dr++; dc--; }
  else if ((dr & 1) == 1 && (dc & 1) == 0) { dr--; dc++; }
  return ((dc >> 1) * m * 2 + dr * 2 + (dc & 1)) * WB + mbyte % WB;
}
// byte offset of metadata byte `mbyte` of row `row` in any of the three storage forms (k = dense columns)
template <int WB>
__host__ __device__ inline int64_t meta_offset(int layout, int64_t mbyte, int64_t row, int64_t m, int64_t k) {
  if (layout == TF24_COMPRESSED_PANEL) return panel_meta_offset(mbyte, row, m);
  if (layout == TF24_COMPRESSED_CUTLASS) return cutlass_meta_offset<WB>(mbyte, row, m);
  return row * (k >> 3) + mbyte;
}

__host__ __device__ inline int dtype_size(int dt) {
  return (dt == TF24_F32 || dt == TF24_I32) ? 4 : (dt == TF24_F16 || dt == TF24_BF16) ? 2 : 1;
}

// ---------------------------------------------------------------- conversions to float (exact)
__device__ __forceinline__ float to_float(float v) { return v; }
__device__ __forceinline__ float to_float(f16_t v) {
  return (float)__builtin_bit_cast(_Float16, v.bits);
}
__device__ __forceinline__ float to_float(bf16_t v) {
  return __builtin_bit_cast(float, (uint32_t)v.bits << 16);
}
__device__ __forceinline__ float to_float(uint8_t v) { return (float)v; }

// ---------------------------------------------------------------- conversions from float
// round-to-nearest-even everywhere, like a plain tensor cast
template <typename T> __device__ __forceinline__ T from_float(float f);
template <> __device__ __forceinline__ float from_float<float>(float f) { return f; }
template <> __device__ __forceinline__ f16_t from_float<f16_t>(float f) {
  return f16_t{__builtin_bit_cast(uint16_t, (_Float16)f)};
}
// gfx950's V_CVT_PK_BF16_F32: round to nearest even, NaNs quieted with their upper payload bits kept --
// on all 2^32 float32 patterns the same bits as the integer sequence (u + 0x7fff + (u >> 16 & 1)) >> 16 with
// (u >> 16) | 0x40 for NaNs, in one instruction per pair instead of seven per value.
template <> __device__ __forceinline__ bf16_t from_float<bf16_t>(float f) {
  return bf16_t{__builtin_bit_cast(uint16_t, (__bf16)f)};
}
// OCP e4m3fn (bias 7, no inf, 0x7f = NaN, max 448): values that round past 448 become NaN,
// exactly like the bit pattern arithmetic of a round-to-nearest-even narrowing.
__host__ __device__ inline uint8_t float_to_e4m3(float f) {
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  uint32_t sign = (u >> 24) & 0x80u;
  u &= 0x7fffffffu;
  uint32_t r;
  if (u >= 0x43f00000u) {            // |f| >= 480, inf, NaN
    r = 0x7fu;
  } else if (u < 0x3c800000u) {      // |f| < 2^-6: subnormal result, multiples of 2^-9
    float a = __builtin_bit_cast(float, u) + 16384.0f;   // ulp(16384) * 2^-23.. aligns 2^-9 to bit 0
    r = __builtin_bit_cast(uint32_t, a) - 0x46800000u;   // 16384.0f == 0x46800000
  } else {
    uint32_t odd = (u >> 20) & 1u;
    u += 0x7ffffu + odd;             // RTNE at bit 20
    r = (u >> 20) - ((127u - 7u) << 3);
  }
  return (uint8_t)(r | sign);
}
// On the device gfx950's V_CVT_PK_FP8_F32 (OCP e4m3fn, round to nearest even, NaN past the range) gives the same
// byte for every float32 pattern that is not a NaN; NaNs take the bit arithmetic's sign | 0x7f (the instruction
// returns 0xff for both signs).  About five instructions instead of twenty.
template <> __device__ __forceinline__ e4m3_t from_float<e4m3_t>(float f) {
  const uint32_t h = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(f, f, 0, false) & 0xffu;
  const uint32_t nan = ((__builtin_bit_cast(uint32_t, f) >> 24) & 0x80u) | 0x7fu;
  return e4m3_t{(uint8_t)(f != f ? nan : h)};
}

__host__ __device__ inline float e4m3_to_float(uint8_t b) {
  uint32_t sign = (uint32_t)(b & 0x80u) << 24;
  uint32_t e = (b >> 3) & 0xfu, m = b & 7u;
  float v;
  if (e == 0) v = (float)m * 0.001953125f;                                    // m * 2^-9
  else if (e == 15 && m == 7) v = __builtin_bit_cast(float, 0x7fc00000u);     // NaN
  else v = __builtin_bit_cast(float, ((e + 120u) << 23) | (m << 20));
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) | sign);
}
__device__ __forceinline__ float to_float(e4m3_t v) { return e4m3_to_float(v.bits); }

// OCP e5m2 (bias 15, infinities, NaN): the upper byte of an IEEE half.  Round to nearest even from
// float32 on the bit pattern: magnitudes of 2^16 and above become infinity (the rounding carries
// 61440..65535 there as well), subnormals (below 2^-14) are rounded by a float32 addition.
__host__ __device__ inline uint8_t float_to_e5m2(float f) {
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  const uint32_t sign = (u >> 24) & 0x80u;
  u &= 0x7fffffffu;
  uint32_t r;
  if (u >= (143u << 23)) {
    r = u > 0x7f800000u ? 0x7fu : 0x7cu;
  } else if (u < (113u << 23)) {
    const float v = __builtin_bit_cast(float, u) + __builtin_bit_cast(float, 134u << 23);
    r = __builtin_bit_cast(uint32_t, v) - (134u << 23);
  } else {
    const uint32_t odd = (u >> 21) & 1u;
    u += ((uint32_t)(15 - 127) << 23) + 0xfffffu + odd;
    r = u >> 21;
  }
  return (uint8_t)(r | sign);
}
// V_CVT_PK_BF8_F32: as above (its NaN is 0x7e | sign; the bit arithmetic's, and torch's, 0x7f | sign)
template <> __device__ __forceinline__ e5m2_t from_float<e5m2_t>(float f) {
  const uint32_t h = (uint32_t)__builtin_amdgcn_cvt_pk_bf8_f32(f, f, 0, false) & 0xffu;
  const uint32_t nan = ((__builtin_bit_cast(uint32_t, f) >> 24) & 0x80u) | 0x7fu;
  return e5m2_t{(uint8_t)(f != f ? nan : h)};
}
// int8: exact for the integers an int8 dense operand holds (the only input the int8 path accepts)
template <> __device__ __forceinline__ i8_t from_float<i8_t>(float f) {
  const float c = f < -128.0f ? -128.0f : (f > 127.0f ? 127.0f : f);
  return i8_t{(uint8_t)(int8_t)(int)c};
}
__device__ __forceinline__ float to_float(i8_t v) { return (float)(int8_t)v.bits; }
__device__ __forceinline__ float to_float(e5m2_t v) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)((uint16_t)v.bits << 8));
}

// ---------------------------------------------------------------- vector loads/stores
template <int BYTES> struct vec_bytes;
template <> struct vec_bytes<2> { using type = uint16_t; };
template <> struct vec_bytes<4> { using type = uint32_t; };
template <> struct vec_bytes<8> { using type = uint2; };
template <> struct vec_bytes<16> { using type = uint4; };
template <> struct vec_bytes<32> { struct alignas(16) type { uint4 a, b; }; };

// load N elements of T (N*sizeof(T) in {2,4,8,16,32} bytes, naturally aligned)
template <typename T, int N>
struct Pack {
  T v[N];
  __device__ __forceinline__ void load(const T* p) {
    using V = typename vec_bytes<sizeof(T) * N>::type;
    *reinterpret_cast<V*>(v) = *reinterpret_cast<const V*>(p);
  }
  __device__ __forceinline__ void store(T* p) const {
    using V = typename vec_bytes<sizeof(T) * N>::type;
    *reinterpret_cast<V*>(p) = *reinterpret_cast<const V*>(v);
  }
  // Streaming variants for data touched once per kernel (non-temporal: the lines are not kept in
  // L2).  On the one-pass conversion kernels they are worth 5-20 %.  Operands that
  // are updated in place gain only where both the load and the store are of this form.
  __device__ __forceinline__ void load_stream(const T* p) {
    constexpr int B = sizeof(T) * N;
    if constexpr (B % 16 == 0) {
      typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
      for (int q = 0; q < B / 16; q++) reinterpret_cast<u32x4*>(v)[q] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p) + q);
    } else if constexpr (B == 8) {
      typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
      *reinterpret_cast<u32x2*>(v) = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(p));
    } else {
      load(p);
    }
  }
  __device__ __forceinline__ void store_stream(T* p) const {
    constexpr int B = sizeof(T) * N;
    if constexpr (B % 16 == 0) {
      typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
      for (int q = 0; q < B / 16; q++) __builtin_nontemporal_store(reinterpret_cast<const u32x4*>(v)[q], reinterpret_cast<u32x4*>(p) + q);
    } else if constexpr (B == 8) {
      typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
      __builtin_nontemporal_store(*reinterpret_cast<const u32x2*>(v), reinterpret_cast<u32x2*>(p));
    } else {
      store(p);
    }
  }
};

// The bytes of 4 adjacent lanes (of a one-dimensional block) as one word, lane 0's lowest, in each of them: data parallel primitives
// move them between lanes without the LDS round trip of a shuffle.
__device__ __forceinline__ uint32_t quad_bytes(uint32_t b) {
  uint32_t w = b << (8 * (threadIdx.x & 3));
  w |= (uint32_t)__builtin_amdgcn_mov_dpp((int)w, 0xb1, 0xf, 0xf, true);      // quad_perm [1,0,3,2]
  w |= (uint32_t)__builtin_amdgcn_mov_dpp((int)w, 0x4e, 0xf, 0xf, true);      // [2,3,0,1]
  return w;
}
// the value of the lane 8 away inside its row of 16 (row_ror:8)
__device__ __forceinline__ uint32_t xor8_lane(uint32_t v) { return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xf, 0xf, true); }

// ---------------------------------------------------------------- 2:4 group math
// The kept elements of one group as four flags, and what the reference's 16-row table
// (_semi_structured_conversions.py:46-82) makes of them: idx0 = 0 if m0, else 1 if m1, else 2;
// idx1 = 1 if m0 & m1 & !m2, else 2 if m2 & (m0 | m1), else 3 -- for any of the 16 flag combinations, not
// only the valid ones with two flags set.  Written on the flags themselves, which the compares leave
// in scalar registers: picking a kept value is two selects on scalar conditions, where the route over
// the packed nibble (bits -> positions -> compares -> three selects per value) costs three times the
// vector instructions.
struct Keep4 {
  bool m0, m1, m2, m3;
  __device__ __forceinline__ bool second_is_1() const { return m0 && m1 && !m2; }
  __device__ __forceinline__ bool second_is_2() const { return m2 && (m0 || m1); }
  template <typename T> __device__ __forceinline__ T first(T v0, T v1, T v2) const { return m0 ? v0 : (m1 ? v1 : v2); }
  template <typename T> __device__ __forceinline__ T second(T v1, T v2, T v3) const { return second_is_1() ? v1 : (second_is_2() ? v2 : v3); }
  // pos0 | pos1 << 2
  __device__ __forceinline__ uint32_t nibble() const {
    const uint32_t lo = m0 ? 0u : (m1 ? 1u : 2u);
    const uint32_t hi = second_is_1() ? 4u : (second_is_2() ? 8u : 12u);
    return lo | hi;
  }
  __device__ __forceinline__ uint32_t bits() const { return (uint32_t)m0 | ((uint32_t)m1 << 1) | ((uint32_t)m2 << 2) | ((uint32_t)m3 << 3); }
};
__device__ __forceinline__ Keep4 keep_from_bits(uint32_t mbits) { return Keep4{(mbits & 1) != 0, (mbits & 2) != 0, (mbits & 4) != 0, (mbits & 8) != 0}; }

// Magnitude mask.  Six strict compares of |x|; ties keep the larger index (all equal -> elements 2 and 3).
__device__ __forceinline__ Keep4 magnitude_keep4(float x0, float x1, float x2, float x3) {
  float a = __builtin_fabsf(x0), b = __builtin_fabsf(x1), c = __builtin_fabsf(x2), d = __builtin_fabsf(x3);
  bool x1_ = a > b, x2_ = a > c, x3_ = a > d, x4_ = b > c, x5_ = b > d, x6_ = c > d;
  Keep4 k;
  k.m0 = (x2_ & x3_) | (x1_ & x2_) | (x1_ & x3_);
  k.m1 = (!x1_ & x5_) | (x4_ & x5_) | (!x1_ & x4_);
  k.m2 = (!x2_ & !x4_) | (!x2_ & x6_) | (!x4_ & x6_);
  k.m3 = (!x3_ & !x5_) | (!x3_ & !x6_) | (!x5_ & !x6_);
  return k;
}
// the same as bits: bit i set = element i kept
__device__ __forceinline__ uint32_t magnitude_mask4(float x0, float x1, float x2, float x3) {
  return magnitude_keep4(x0, x1, x2, x3).bits();
}

// mask bits -> nibble pos0 | pos1<<2 (the 16-row table: masks with other than two bits set
// are mapped as the reference's boolean minimisation maps them)
__device__ __forceinline__ uint32_t encode_nibble(uint32_t mbits) { return keep_from_bits(mbits).nibble(); }

// Magnitude selection of one group of four 16-bit floats (f16 or bf16) held as two dwords
// (x1:x0, x3:x2), in integer arithmetic: for numbers the order of |x| is the order of the low 15
// bits, so key_i = |bits_i| << 2 | i orders the elements by (|x|, index) -- exactly the rule of the
// six compares (a tie keeps the larger index) -- and the two kept elements are the largest and the
// second largest key: four min/max pairs, a max and a max3.  Returns the nibble pos0 | pos1 << 2;
// `top_key` (largest key) lets the caller test for NaN, whose magnitude bits lie above infinity's:
// a group with a NaN follows the float compares instead (NaN compares false either way there).
// About 20 instructions against about 60 for compares, lane-mask logic and the table encoding.
struct Top2 { uint32_t nibble, top_key; };
__device__ __forceinline__ Top2 magnitude_top2_16(uint32_t lo, uint32_t hi) {
  const uint32_t k0 = (lo & 0x7fffu) << 2;
  const uint32_t k1 = (((lo >> 16) & 0x7fffu) << 2) | 1u;
  const uint32_t k2 = ((hi & 0x7fffu) << 2) | 2u;
  const uint32_t k3 = (((hi >> 16) & 0x7fffu) << 2) | 3u;
  const uint32_t hi01 = max(k0, k1), lo01 = min(k0, k1), hi23 = max(k2, k3), lo23 = min(k2, k3);
  const uint32_t top = max(hi01, hi23);
  const uint32_t second = max(min(hi01, hi23), max(lo01, lo23));
  const uint32_t p = top & 3u, q = second & 3u;
  return {min(p, q) | (max(p, q) << 2), top};
}
// the 16-bit element at position pos (0..3) of the group (x1:x0, x3:x2), in the low half of the result
__device__ __forceinline__ uint32_t pick16(uint32_t lo, uint32_t hi, uint32_t pos) {
  const uint64_t both = ((uint64_t)hi << 32) | lo;
  return (uint32_t)(both >> (pos << 4));
}

template <typename T>
__device__ __forceinline__ T select4(uint32_t pos, T v0, T v1, T v2, T v3) {
  T lo = (pos & 1) ? v1 : v0;
  T hi = (pos & 1) ? v3 : v2;
  return (pos & 2) ? hi : lo;
}

// Float32 division for operands inside the normal range, correctly rounded in five instructions (a reciprocal can be
// shared by several quotients).
//   refined_rcp: one Newton step on v_rcp_f32.  On gfx950 the result is RN(1/b) for every b from 2^-126 up to 2^126
//     (all 2.1e9 bit patterns compared with 1/b in float64).
//   div_in_range: q = RN(a r), then ONE residual correction.  With a, b in [1, 2) and r = RN(1/b), q is off by less
//     than a/2 + 1/2 units in its last place when a < b and by less than 1 when a >= b.  A quotient of two 24-bit
//     numbers is never closer than 2^-25 units to a midpoint between two floats (the distance is a non-zero multiple of
//     1/(2B), B < 2^24 the integer of b), and beside a midpoint q is therefore off by half a unit (one and a half would
//     take a = 2 - 2^-23 < b < 2).  There the residual is exact and the corrected sum, before its one rounding, is off by
//     at most 2^-25 b/2 < 2^-25 units: it rounds as the quotient does.  (Compared with the float64 quotient on 1e11
//     random and adversarial pairs; the general sequence takes a second correction because it does not assume r.)
// Needed: numerator and denominator normal, |numerator| > 2^-104, denominator < 2^126, exponent difference below 96
// and a normal quotient.  Callers establish those bounds and use operator/ outside them.
__device__ __forceinline__ float refined_rcp(float b) {
  float r = __builtin_amdgcn_rcpf(b);
  return __builtin_fmaf(__builtin_fmaf(-b, r, 1.0f), r, r);
}
__device__ __forceinline__ float div_in_range(float a, float b, float r) {
  const float q = a * r;
  return __builtin_fmaf(__builtin_fmaf(-b, q, a), r, q);
}

// Counter-based uniforms for MVUE24 when no tensor is supplied: Philox4x32-10 (Salmon et al., the
// generator of Random123 / cuRAND / torch), key = seed, counter = {index, offset}.  One call gives
// the four uniforms of two adjacent groups: `index` = row * (k / 8) + (8-column unit of the row),
// words 0,1 for the even group of the unit and 2,3 for the odd one.
struct Philox4 { uint32_t x, y, z, w; };
// The calls for the counters index, index + stride, ... of one lane.  The only generator here: uniforms that are written out are those that a
// conversion draws, and saved seeds have to give the same bits as ever (the oracle has its own, pinned by known answers).  With
// three-input exclusive ors (v_bitop3_b32) a call takes 40 + 2 vector instructions instead of 58, which is what kernels that sample are bound
// by (see mvue4).
template <int N>
__device__ __forceinline__ void philox4x32_10_calls(uint64_t seed, uint64_t index, uint64_t stride, uint64_t offset, Philox4 (&out)[N]) {
  uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
#pragma unroll
  for (int i = 0; i < N; i++) {
    const uint64_t at = index + (uint64_t)i * stride;
    out[i] = Philox4{(uint32_t)at, (uint32_t)(at >> 32), (uint32_t)offset, (uint32_t)(offset >> 32)};
  }
#pragma unroll
  for (int round = 0; round < 10; round++) {
#pragma unroll
    for (int i = 0; i < N; i++) {
      const uint64_t p0 = (uint64_t)0xD2511F53u * out[i].x, p1 = (uint64_t)0xCD9E8D57u * out[i].z;
      const uint32_t h0 = (uint32_t)(p0 >> 32), h1 = (uint32_t)(p1 >> 32);
      if (round == 0) out[i] = Philox4{out[i].y ^ (h1 ^ k0), (uint32_t)p1, h0 ^ (out[i].w ^ k1), (uint32_t)p0};   // (the offset's words are the same in all lanes)
      else out[i] = Philox4{(uint32_t)__builtin_amdgcn_bitop3_b32(h1, out[i].y, k0, 0x96), (uint32_t)p1,
                            (uint32_t)__builtin_amdgcn_bitop3_b32(h0, out[i].w, k1, 0x96), (uint32_t)p0};
    }
    k0 += 0x9E3779B9u; k1 += 0xBB67AE85u;
  }
}
// 24 random bits -> [0, 1), exact in float32
__host__ __device__ inline float philox_uniform(uint32_t bits) { return (float)(bits & 0xffffffu) * 5.9604644775390625e-8f; }

// Where MVUE24 takes its uniforms from
enum { RAND_FULL = 0, RAND_PACKED = 1, RAND_SEEDED = 2 };
struct RandSrc {
  const float* ptr;       // RAND_FULL: [m, k] (columns 4g, 4g+1 used); RAND_PACKED: [m, k/2]
  int64_t ld;
  int kind;
  uint64_t seed, offset;  // RAND_SEEDED
  const uint64_t* state;  // RAND_SEEDED: when not null, {seed, offset} are read from here (device memory) by the kernel
  __device__ __forceinline__ uint64_t seed_now() const { return state ? state[0] : seed; }
  __device__ __forceinline__ uint64_t offset_now() const { return state ? state[1] : offset; }
};

// MVUE24 of one group in float32, in the reference's operation order (no contraction): inclusion
// probabilities p_i, the kept elements, and the two kept values x_i / p_i in ascending position.  Only the two kept
// values are divided.
struct Mvue4 {
  uint32_t nibble, bits;      // of the kept flags (as words: flags merged behind a branch would be rebuilt from registers)
  float first, second;
};

// FAST: every division through div_in_range, in straight-line code; `ok` says whether the bounds of div_in_range held
// throughout (if not, the result is not to be used).  |x_i| + eps >= 2^-23 always, so with sum < 2^40 and every
// s_i = sum - a_i > 0 (then s_i >= 2^-46) the quotients t_i = a_i/sum >= 2^-63 and k_i = t_i/s_i >= 2^-104 meet them;
// p_i >= t_i because k >= k_i for a rounded sum of non-negatives, so p_i in [2^-63, 4] once two of them add up to at most 4, and
// |x_i| <= sum p_i keeps the exponents within 96 of each other; |x_i| >= 2^-100 or x_i = 0 keeps the quotient normal or
// zero.  (Half precision, WIDE = false, holds neither a sum of 2^40 nor a value below 2^-100.)
template <bool FAST, bool WIDE>
__device__ __forceinline__ Mvue4 mvue4_as(const float (&x)[4], float r0, float r1, bool& ok) {
  const float eps = 1.19209e-07f;
  const float a0 = __builtin_fabsf(x[0]) + eps, a1 = __builtin_fabsf(x[1]) + eps;
  const float a2 = __builtin_fabsf(x[2]) + eps, a3 = __builtin_fabsf(x[3]) + eps;
  const float sum = ((a0 + a1) + a2) + a3;
  const float s0 = sum - a0, s1 = sum - a1, s2 = sum - a2, s3 = sum - a3;
  float t0, t1, t2, t3, k0, k1, k2, k3;
  if constexpr (FAST) {
    const float rs = refined_rcp(sum);
    t0 = div_in_range(a0, sum, rs); t1 = div_in_range(a1, sum, rs);
    t2 = div_in_range(a2, sum, rs); t3 = div_in_range(a3, sum, rs);
    k0 = div_in_range(t0, s0, refined_rcp(s0)); k1 = div_in_range(t1, s1, refined_rcp(s1));
    k2 = div_in_range(t2, s2, refined_rcp(s2)); k3 = div_in_range(t3, s3, refined_rcp(s3));
  } else {
    t0 = a0 / sum; t1 = a1 / sum; t2 = a2 / sum; t3 = a3 / sum;
    k0 = t0 / s0; k1 = t1 / s1; k2 = t2 / s2; k3 = t3 / s3;
  }
  const float k = ((k0 + k1) + k2) + k3;
  const float p0 = t0 + a0 * (k - k0), p1 = t1 + a1 * (k - k1), p2 = t2 + a2 * (k - k2), p3 = t3 + a3 * (k - k3);
  // (FAST: no term is negative, nor a NaN unless `ok` fails, so each compare implies the next one, and "this and none before" is
  // where two neighbours differ; a condition that is used negated as well costs a second compare)
  const bool m0 = r0 <= t0, upto1 = r0 <= (t0 + t1), upto2 = r0 <= ((t0 + t1) + t2);
  const bool m1 = FAST ? upto1 != m0 : upto1 && !m0;
  const bool m2 = FAST ? upto2 != upto1 : upto2 && !m1 && !m0;
  const bool m3 = FAST ? !upto2 : !m2 && !m1 && !m0;
  const float d0 = m0 ? 0.0f : a0, d1 = m1 ? 0.0f : a1, d2 = m2 ? 0.0f : a2;
  const float d3 = FAST ? (upto2 ? a3 : 0.0f) : (m3 ? 0.0f : a3);
  const float dsum = ((d0 + d1) + d2) + d3;
  const float t = r1 * dsum;
  const bool e0 = t <= d0, to1 = t <= (d0 + d1), to2 = t <= ((d0 + d1) + d2);
  const bool e1 = FAST ? to1 != e0 : to1 && !e0;
  const bool e2 = FAST ? to2 != to1 : to2 && !e1 && !e0;
  const bool e3 = FAST ? !to2 : !e2 && !e1 && !e0;
  const Keep4 keep{m0 || e0, m1 || e1, m2 || e2, m3 || e3};
  const float xa = keep.first(x[0], x[1], x[2]), xb = keep.second(x[1], x[2], x[3]);
  const float pa = keep.first(p0, p1, p2), pb = keep.second(p1, p2, p3);
  Mvue4 g;
  g.nibble = keep.nibble();
  g.bits = keep.bits();
  if constexpr (FAST) {
    // div_in_range with the residual's sign turned round, which keeps the sign of a zero numerator
    const float ra = refined_rcp(pa), rb = refined_rcp(pb);
    const float qa = xa * ra, qb = xb * rb;
    g.first = __builtin_fmaf(-__builtin_fmaf(pa, qa, -xa), ra, qa);
    g.second = __builtin_fmaf(-__builtin_fmaf(pb, qb, -xb), rb, qb);
    // an s_i of zero (they are never negative) makes its reciprocal, k and with it every p a NaN: no test of its own
    ok = pa + pb <= 4.0f;
    if constexpr (WIDE) {        // In can hold what half precision cannot: a sum of 2^40, values below 2^-100
      ok = ok && sum < 0x1p40f;
      // 0 or at least 2^-100 (0x0d800000), for both, twice without the sign: one less than zero wraps round
      const uint32_t ua = (__builtin_bit_cast(uint32_t, xa) << 1) - 1u, ub = (__builtin_bit_cast(uint32_t, xb) << 1) - 1u;
      ok = ok && (ua < ub ? ua : ub) >= 2u * 0x0d800000u - 1u;
    }
  } else {
    g.first = xa / pa;
    g.second = xb / pb;
    ok = true;
  }
  return g;
}

// What bounds the kernels that call this, when the uniforms are drawn in the kernel, is the number of their vector instructions:
// with eight waves on a SIMD one issues every 2.6 cycles on average (counters of an 8192 x 8192 conversion), and although by
// themselves float32 arithmetic and bitwise operations issue at up to twice the rate of compares, selects, minima and conversions, and
// at half of it with an operand in a scalar register, a mixture follows the count (keys and constants moved to vector registers
// for the faster rate, one instruction more each: no gain).  A group costs 116 of them, a generator call 42 for two groups.  One correction per division instead of two, no
// branch and one test of the bounds per group (the slow path is laid out behind the kernel), flags as short-circuit
// expressions (as integers they went through vector registers), kept values converted without a test for NaN, and leaner
// addresses in the callers: 8192 x 8192 bf16 to e4m3 82 -> 64.5 us, to fp16 78.6 -> 64.5 (with a supplied tensor its
// 268 MB are the bound: 80 us before and after), a column-major 3072 x 12288 half matrix with its row sums 54.5 -> 44 us.
// Three-input exclusive ors, six compares instead of nine and a kernel of its own for panel output, on another card: 60.5 -> 54.9,
// 61.5 -> 57.0 and 37.1 -> 36.1.  Each taken back by itself, 8192 x 8192 bf16 to fp16, to e4m3, float32 to fp16 (58.7, 56.9, 65.6 with
// all): the exclusive ors 60.7, 60.2, 67.9, the compares 60.5, 59.7, 66.9, the kernel 61.1, 61.1, 67.7; the shorter range tests 58.8, 59.4, 65.3
// (one median of three beyond the spread), the bytes of a quad in two steps instead of three 58.3, 57.7, 65.9 (none, nor in the modes bound by memory).
template <typename In>
__device__ __forceinline__ Mvue4 mvue4(const float (&x)[4], float r0, float r1, bool& finite) {
  bool ok;
  Mvue4 g = mvue4_as<true, !std::is_same<In, f16_t>::value>(x, r0, r1, ok);
  finite = ok;
  if (__builtin_expect(!ok, 0)) g = mvue4_as<false, false>(x, r0, r1, ok);
  return g;
}

// Two values next to each other as they are stored, `finite`: neither is a NaN (spares the 8-bit types the test).
template <typename Out>
__device__ __forceinline__ Pack<Out, 2> from_float2(float a, float b, bool finite) {
  Pack<Out, 2> o;
  if constexpr (std::is_same<Out, e4m3_t>::value || std::is_same<Out, e5m2_t>::value) {
    uint32_t w;
    if constexpr (std::is_same<Out, e4m3_t>::value) w = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
    else w = (uint32_t)__builtin_amdgcn_cvt_pk_bf8_f32(a, b, 0, false);
    if (__builtin_expect(!finite, 0)) w = (uint32_t)from_float<Out>(a).bits | ((uint32_t)from_float<Out>(b).bits << 8);
    o.v[0].bits = (uint8_t)w;
    o.v[1].bits = (uint8_t)(w >> 8);
  } else {
    o.v[0] = from_float<Out>(a);
    o.v[1] = from_float<Out>(b);
  }
  return o;
}

// Four values, two of either group; 8-bit types in one word, the second pair converted into its upper half.
template <typename Out>
__device__ __forceinline__ Pack<Out, 4> from_float4(float a0, float b0, bool finite0, float a1, float b1, bool finite1) {
  Pack<Out, 4> o;
  if constexpr (std::is_same<Out, e4m3_t>::value || std::is_same<Out, e5m2_t>::value) {
    int w;
    asm("" : "=v"(w));                           // (what the conversions leave alone is written by the other one)
    if constexpr (std::is_same<Out, e4m3_t>::value) w = __builtin_amdgcn_cvt_pk_fp8_f32(a1, b1, __builtin_amdgcn_cvt_pk_fp8_f32(a0, b0, w, false), true);
    else w = __builtin_amdgcn_cvt_pk_bf8_f32(a1, b1, __builtin_amdgcn_cvt_pk_bf8_f32(a0, b0, w, false), true);
    if (__builtin_expect(!(finite0 && finite1), 0))
      w = (int)((uint32_t)from_float<Out>(a0).bits | ((uint32_t)from_float<Out>(b0).bits << 8) | ((uint32_t)from_float<Out>(a1).bits << 16) | ((uint32_t)from_float<Out>(b1).bits << 24));
    __builtin_memcpy(o.v, &w, 4);
  } else {
    o.v[0] = from_float<Out>(a0); o.v[1] = from_float<Out>(b0);
    o.v[2] = from_float<Out>(a1); o.v[3] = from_float<Out>(b1);
  }
  return o;
}

// ---------------------------------------------------------------- LDS within a wave
// Between what the lanes of one wave write to LDS and what others of its lanes read there, either way round: no instruction, the LDS accesses of a
// wave execute in order.  It keeps the compiler to that order, to which the accesses of one lane at different addresses have none (a scheduling barrier
// binds the instruction scheduler, not the passes before it).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------- row sums
// out[r] = sum over column blocks of partial[b * m + r], one rounding to out's type (F32 | F16 | BF16): what is left to do behind a
// conversion that also adds the rows of its matrix, 128 columns at a time.
struct RowSums {
  const float* partial;
  int nblocks;
  int64_t m;
  void* out;
  int dtype;
  int64_t blocks() const { return (m + 31) / 32; }
};
// Rows 32 `block` .. + 31, by the first 256 lanes of a workgroup (all of which enter).  8 groups of 32 lanes each add every 8th column
// block (coalesced 128-byte reads), then the 8 group sums of a row are added in group order.
__device__ __forceinline__ void row_sums_of_block(const RowSums& s, int64_t block) {
  __shared__ float s_part[8][32];
  const int lr = threadIdx.x & 31, part = threadIdx.x >> 5;
  const int64_t r = block * 32 + lr;
  float t = 0.0f;
  if (r < s.m && part < 8) {
    // eight loads in flight: waiting for each made this tail 5 us long on 96 column blocks
    for (int b = part; b < s.nblocks; b += 64) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; u++) v[u] = b + 8 * u < s.nblocks ? s.partial[(int64_t)(b + 8 * u) * s.m + r] : 0.0f;
#pragma unroll
      for (int u = 0; u < 8; u++) t += v[u];
    }
  }
  if (part < 8) s_part[part][lr] = t;
  __syncthreads();
  if (part == 0 && r < s.m) {
    float sum = 0.0f;
#pragma unroll
    for (int q = 0; q < 8; q++) sum += s_part[q][lr];
    if (s.dtype == TF24_F32) reinterpret_cast<float*>(s.out)[r] = sum;
    else if (s.dtype == TF24_F16) reinterpret_cast<f16_t*>(s.out)[r] = from_float<f16_t>(sum);
    else reinterpret_cast<bf16_t*>(s.out)[r] = from_float<bf16_t>(sum);
  }
}
// The conversion of a column-major matrix by an MVUE mode that draws its uniforms, to panel form of the same 16-bit type, its partial
// sums left in `partial`; and the launch that finishes them.
int compress_with_partial_sums(const char* fn, const void* dense, int dtype, int64_t ld, int64_t m, int64_t k, int mode, const void* rnd, void* values, void* meta,
                               float* partial, hipStream_t stream);
int finish_row_sums(const char* fn, const RowSums& sums, hipStream_t stream);

}  // namespace tf24
