// 2:4 sparse x dense matmul on the gfx950 sparse matrix cores (V_SMFMAC), float32 accumulation.
//
//     C[i,j] = act( scale * sum_k A[i,k] * B(k,j) + bias[i] )
//
// A is the compressed operand (values [n_sparse, k/2] + canonical metadata), which is exactly the
// SMFMAC "A" operand: one lane holds a run of consecutive compressed values of one row and the
// matching run of 2-bit positions is a contiguous slice of the row's metadata stream.
//
// Operand layouts of the instructions used (R = 16 or 32 rows, lane l, nkb = 64/R lane blocks,
// K dense depth of the instruction, kper = K/nkb):
//   A: row l%R, block ka = l/R holds the kper/2 compressed values of dense k in [ka*kper, (ka+1)*kper);
//      value e uses index bits [2e+1:2e] (16-bit types: the 16-bit half of the index register
//      selected by ABID; 8-bit types: all 32 bits)
//   B: column l%R, block kb = l/R holds dense k in [kb*kper/2, (kb+1)*kper/2) followed by the same
//      range shifted by K/2
//   D: 16x16: column l%16, rows 4*(l/16)+r;  32x32: column l%32, rows 8*(r/4) + 4*(l/32) + r%4
#pragma once
#include "lds_copies.hpp"
#include <algorithm>
#include <type_traits>

namespace tf24 {
namespace {

typedef _Float16 half16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x16 __attribute__((ext_vector_type(16)));
typedef int int8v __attribute__((ext_vector_type(8)));
typedef int int16v __attribute__((ext_vector_type(16)));

// ---- element traits: KSTEP = dense depth of one 16x16 instruction; all types move 64 bytes of
// compressed A and 128 bytes of B per row per step.
template <typename T> struct mma16;
template <> struct mma16<f16_t> {
  static constexpr int KSTEP = 64;
  using acc_t = float4v;
  template <int ABID>
  static __device__ __forceinline__ float4v run(int4v a, int8v b, float4v c, int idx) {
    return __builtin_amdgcn_smfmac_f32_16x16x64_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half16, b), c, idx, 0, ABID);
  }
};
template <> struct mma16<bf16_t> {
  static constexpr int KSTEP = 64;
  using acc_t = float4v;
  template <int ABID>
  static __device__ __forceinline__ float4v run(int4v a, int8v b, float4v c, int idx) {
    return __builtin_amdgcn_smfmac_f32_16x16x64_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x16, b), c, idx, 0, ABID);
  }
};
template <> struct mma16<e4m3_t> {
  static constexpr int KSTEP = 128;
  using acc_t = float4v;
  template <int ABID>
  static __device__ __forceinline__ float4v run(int4v a, int8v b, float4v c, int idx) {
    return __builtin_amdgcn_smfmac_f32_16x16x128_fp8_fp8(a, b, c, idx, 0, 0);
  }
};
template <> struct mma16<e5m2_t> {
  static constexpr int KSTEP = 128;
  using acc_t = float4v;
  template <int ABID>
  static __device__ __forceinline__ float4v run(int4v a, int8v b, float4v c, int idx) {
    return __builtin_amdgcn_smfmac_f32_16x16x128_bf8_bf8(a, b, c, idx, 0, 0);
  }
};

template <> struct mma16<i8_t> {
  static constexpr int KSTEP = 128;
  using acc_t = int4v;
  template <int ABID>
  static __device__ __forceinline__ int4v run(int4v a, int8v b, int4v c, int idx) {
    return __builtin_amdgcn_smfmac_i32_16x16x128_i8(a, b, c, idx, 0, 0);
  }
};

// Exact (erf) GELU, 0.5 v (1 + erf(v / sqrt 2)), through the complementary error function of |v| / sqrt 2
// (Abramowitz & Stegun 7.1.26: erfc(z) = t (a1 + t (a2 + t (a3 + t (a4 + t a5)))) exp(-z^2), t = 1 / (1 + p z),
// absolute error <= 1.5e-7):  with q = erfc(|v| / sqrt 2),  gelu(v) = v - v q / 2 for v >= 0 and v q / 2 below,
// so the negative tail is not formed as a difference of nearly equal numbers.  One reciprocal, one exponential
// and nine multiply-adds per element: the library erff costs three times that, which made a GELU output pass
// slower than a plain one plus a separate GELU kernel.  Agrees with the float32 GELU of torch to 3e-7 absolute.
__device__ __forceinline__ float gelu_erf(float v) {
  const float z = __builtin_fabsf(v) * 0.70710678118654752f;
  const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.3275911f, z, 1.0f));
  float poly = __builtin_fmaf(t, 1.061405429f, -1.453152027f);
  poly = __builtin_fmaf(poly, t, 1.421413741f);
  poly = __builtin_fmaf(poly, t, -0.284496736f);
  poly = __builtin_fmaf(poly, t, 0.254829592f);
  const float q = poly * t * __builtin_amdgcn_exp2f(z * z * -1.4426950408889634f);
  // |v| clamped where q has long been 0: an infinite v stays infinite (or becomes -0) instead of inf * 0
  const float h = 0.5f * q * __builtin_amdgcn_fmed3f(v, -65536.0f, 65536.0f);
  return v >= 0.0f ? v - h : (v < 0.0f ? h : v);
}

__device__ __forceinline__ float apply_act(float v, int act) {
  act &= ~TF24_BIAS_F32;
  if (act == TF24_ACT_RELU) return v > 0.0f ? v : 0.0f;
  if (act == TF24_ACT_SILU) return v / (1.0f + __expf(-v));
  if (act == TF24_ACT_GELU) return gelu_erf(v);
  return v;
}

// An accumulator element -> the finished output element.  Floating accumulators: scale, bias,
// activation, one rounding.  Integer accumulators (int8 operands): bias and ReLU in int32, exact.
template <typename OutT> __device__ __forceinline__ OutT to_out(float v) { return from_float<OutT>(v); }
template <typename OutT> __device__ __forceinline__ OutT to_out(int v) { return (OutT)v; }
template <typename OutT>
__device__ __forceinline__ float finish_value(float accv, float scale, const OutT* bias, int64_t row, int act) {
  float v = accv * scale;
  if (bias) {
    if (sizeof(OutT) == 2 && (act & TF24_BIAS_F32)) v += to_float(from_float<OutT>(reinterpret_cast<const float*>(bias)[row]));
    else v += to_float(bias[row]);
  }
  return apply_act(v, act);
}
template <typename OutT>
__device__ __forceinline__ int finish_value(int accv, float, const OutT* bias, int64_t row, int act) {
  int v = accv;
  if (bias) v += (int)bias[row];
  return (act == TF24_ACT_RELU && v < 0) ? 0 : v;
}

// The output pass of the tiled kernel is compiled once per epilogue: plain, bias only, and bias (or none) followed by
// each activation.  Left to run-time tests alone, the per-element selects and the inlined SiLU more than triple the
// time of the pass (21 000 against 6 300 cycles per 256 x 256 tile), which is a tenth of the whole kernel at k = 4096.
// The bias of an element arrives as a value: the pass reads it from LDS, where the wave has put the bias of its rows
// (zeros without one).
enum { EPI_PLAIN = 0, EPI_BIAS = 1, EPI_RELU = 2, EPI_SILU = 3, EPI_GELU = 4 };
template <int MODE>
__device__ __forceinline__ float finish_element(float accv, float scale, float biasv) {
  float v = accv * scale;
  if constexpr (MODE != EPI_PLAIN) v += biasv;
  if constexpr (MODE == EPI_RELU) v = v > 0.0f ? v : 0.0f;
  if constexpr (MODE == EPI_SILU) v = v * __builtin_amdgcn_rcpf(1.0f + __expf(-v));   // (1 ulp reciprocal: the IEEE division is 10 instructions)
  if constexpr (MODE == EPI_GELU) v = gelu_erf(v);
  return v;
}
// integer accumulators: bias and ReLU in int32, exact (the other activations are not defined for them)
template <int MODE>
__device__ __forceinline__ int finish_element(int accv, float, int biasv) {
  int v = accv;
  if constexpr (MODE != EPI_PLAIN) v += biasv;
  if constexpr (MODE == EPI_RELU) v = v < 0 ? 0 : v;
  return v;
}
template <typename OutT> __device__ __forceinline__ float bias_as(float, OutT b) { return to_float(b); }
template <typename OutT> __device__ __forceinline__ int bias_as(int, OutT b) { return (int)b; }
// a bias element as the bits its load leaves in a register, and back
template <typename OutT> __device__ __forceinline__ uint32_t bias_bits(OutT b) {
  if constexpr (sizeof(OutT) == 2) { uint16_t h; __builtin_memcpy(&h, &b, 2); return h; }
  else { uint32_t w; __builtin_memcpy(&w, &b, 4); return w; }
}
template <typename OutT> __device__ __forceinline__ OutT bias_from_bits(uint32_t w) {
  OutT b;
  if constexpr (sizeof(OutT) == 2) { const uint16_t h = (uint16_t)w; __builtin_memcpy(&b, &h, 2); }
  else __builtin_memcpy(&b, &w, 4);
  return b;
}

// ------------------------------------------------------------------------------------------
// General kernel: operands straight from global memory (cached), every supported shape and
// layout.  One wave computes a 32(i) x 32(j) tile with 16x16 instructions; a block is 2x2 waves.
// ------------------------------------------------------------------------------------------
template <typename T, typename OutT, bool B_KCONTIG, bool C_JMAJOR>
__global__ void __launch_bounds__(256)
spmm_general(const uint8_t* __restrict__ a_values, const uint8_t* __restrict__ a_meta, int64_t n_sparse, int64_t k,
             const T* __restrict__ b, int64_t ldb, int64_t n_dense,
             OutT* __restrict__ c, int64_t ldc, const OutT* __restrict__ bias, float scale, int act, int a_layout) {
  constexpr int KSTEP = mma16<T>::KSTEP;
  const bool panel = a_layout == TF24_COMPRESSED_PANEL;
  constexpr int ES = sizeof(T);                       // element size of values and B
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t i0 = (int64_t)blockIdx.y * 64 + (wave >> 1) * 32;
  const int64_t j0 = (int64_t)blockIdx.x * 64 + (wave & 1) * 32;
  if (i0 >= n_sparse || j0 >= n_dense) return;       // whole wave out of range
  const int li = lane & 15, lk = lane >> 4;
  const int64_t a_pitch = (k / 2) * ES;               // bytes per row of compressed values
  typename mma16<T>::acc_t acc[2][2];
#pragma unroll
  for (int ti = 0; ti < 2; ti++)
#pragma unroll
    for (int tj = 0; tj < 2; tj++)
#pragma unroll
      for (int r = 0; r < 4; r++) acc[ti][tj][r] = 0;

  for (int64_t k0 = 0; k0 < k; k0 += KSTEP) {
    int4v af[2];
    int idx[2];
#pragma unroll
    for (int ti = 0; ti < 2; ti++) {
      const int64_t row = i0 + ti * 16 + li;
      // one instruction step is exactly one panel of values (KSTEP dense columns: 64 value bytes); the lane's
      // index word is metadata bytes k0/8 + lk*2.. (16-bit values) or k0/8 + lk*4.. (8-bit) of its row
      const int64_t voff = panel ? ((k0 / KSTEP) * n_sparse + row) * 64 : row * a_pitch + (k0 / 2) * ES;
      const int64_t mbyte = k0 / 8 + lk * (ES == 2 ? 2 : 4);
      const int64_t moff = meta_offset<ES == 2 ? 2 : 4>(a_layout, mbyte, row, n_sparse, k);   // (reordered metadata: the reference's own storage)
      af[ti] = *reinterpret_cast<const int4v*>(a_values + voff + lk * 16);
      if constexpr (ES == 2) idx[ti] = *reinterpret_cast<const uint16_t*>(a_meta + moff);
      else idx[ti] = *reinterpret_cast<const int*>(a_meta + moff);
    }
    int8v bf[2];
#pragma unroll
    for (int tj = 0; tj < 2; tj++) {
      int64_t col = j0 + tj * 16 + li;
      if (col >= n_dense) col = n_dense - 1;          // clamp: the column is never stored
      constexpr int HALF = KSTEP / 8;                 // elements per half run (16 bytes)
      if constexpr (B_KCONTIG) {
        const T* p = b + col * ldb + k0 + lk * HALF;
        int4v lo = *reinterpret_cast<const int4v*>(p);
        int4v hi = *reinterpret_cast<const int4v*>(p + KSTEP / 2);
        bf[tj] = int8v{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      } else {
        alignas(32) T tmp[2 * HALF];
#pragma unroll
        for (int e = 0; e < HALF; e++) {
          tmp[e] = b[(k0 + lk * HALF + e) * ldb + col];
          tmp[HALF + e] = b[(k0 + KSTEP / 2 + lk * HALF + e) * ldb + col];
        }
        bf[tj] = *reinterpret_cast<int8v*>(tmp);
      }
    }
#pragma unroll
    for (int ti = 0; ti < 2; ti++)
#pragma unroll
      for (int tj = 0; tj < 2; tj++) acc[ti][tj] = mma16<T>::template run<0>(af[ti], bf[tj], acc[ti][tj], idx[ti]);
  }

#pragma unroll
  for (int ti = 0; ti < 2; ti++)
#pragma unroll
    for (int tj = 0; tj < 2; tj++) {
      const int64_t col = j0 + tj * 16 + li;
      if (col >= n_dense) continue;
      const int64_t row = i0 + ti * 16 + lk * 4;
      OutT o[4];
#pragma unroll
      for (int r = 0; r < 4; r++) o[r] = to_out<OutT>(finish_value(acc[ti][tj][r], scale, bias, row + r, act));
      if constexpr (C_JMAJOR) {
        *reinterpret_cast<Pack<OutT, 4>*>(c + col * ldc + row) = *reinterpret_cast<Pack<OutT, 4>*>(o);
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++) c[(row + r) * ldc + col] = o[r];
      }
    }
}


// ------------------------------------------------------------------------------------------
// Tiled kernel: A in the panel layout, B with k contiguous.
//
// A block computes a 256(i) x 256(j) tile (or one of the other TileCfgT shapes) with V_SMFMAC_F32_32X32X32_{F16,BF16} / 32X32X64_FP8:
// 8 waves (2 along i x 4 along j), wave tile 128 x 64 = 4 x 2 instructions, 2 waves per SIMD.
// (4 waves with 128 x 128 wave tiles and 256 accumulators read less LDS per instruction but were
// measured slower: with one wave per SIMD nothing covers a wave's own stalls.)
// Operands go global -> LDS directly (GLOBAL_LOAD_LDS_DWORDX4: lane l of a wave writes
// LDS[base + 16*l], a wave fills 1 KB of contiguous LDS) through a ring of three stage buffers of
// 128 bytes of dense k per row (two instruction steps): while stage s is multiplied, the copies of
// stages s+1 and s+2 are in flight.  LDS rows are unpadded; bank conflicts are avoided by
// XOR-swizzling the 16-byte chunk index with row bits (B: chunk ^ ((row>>1)&7) in 128-byte rows,
// A: chunk ^ ((row>>2)&3) in 64-byte rows), applied on the global side of the copy and again in the
// fragment reads.  The three buffers are slices of one LDS array addressed by a rotating
// wave-uniform offset; the copies are written in assembly the compiler does not look into, so the
// only LDS accesses it sees in the main loop are fragment reads.
// Workgroup ids are remapped so that the 8 XCDs (ids are dealt round-robin) each walk a
// contiguous range of tiles in an 8-tile-high grouped raster: the ~32 tiles resident on an XCD
// form an 8 x 4 patch that shares A rows and B columns in that XCD's L2.
// With more tiles than compute units (and no k pieces) one workgroup per compute unit walks its
// tiles in one pipeline (PERSIST): the copies of the next tile's first two stages ride in the last
// two stages of the current one, and the output pass stages through the one buffer that is free.
// At sustained clocks this kernel runs against the board's power limit (the shader clock settles
// well below its 2.4 GHz maximum, the lower the more the operand bits toggle): what buys time is
// fewer bytes moved per instruction, not a tighter schedule.
// ------------------------------------------------------------------------------------------
template <typename T> struct mma32;
template <> struct mma32<f16_t> {
  using acc_t = float16v;
  using acc4_t = float4v;
  static __device__ __forceinline__ float16v run(int4v a, int8v b, float16v c, int idx) {
    return __builtin_amdgcn_smfmac_f32_32x32x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half16, b), c, idx, 0, 0);
  }
};
template <> struct mma32<bf16_t> {
  using acc_t = float16v;
  using acc4_t = float4v;
  static __device__ __forceinline__ float16v run(int4v a, int8v b, float16v c, int idx) {
    return __builtin_amdgcn_smfmac_f32_32x32x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x16, b), c, idx, 0, 0);
  }
};
template <> struct mma32<e4m3_t> {
  using acc_t = float16v;
  using acc4_t = float4v;
  static __device__ __forceinline__ float16v run(int4v a, int8v b, float16v c, int idx) {
    return __builtin_amdgcn_smfmac_f32_32x32x64_fp8_fp8(a, b, c, idx, 0, 0);
  }
};
template <> struct mma32<e5m2_t> {
  using acc_t = float16v;
  using acc4_t = float4v;
  static __device__ __forceinline__ float16v run(int4v a, int8v b, float16v c, int idx) {
    return __builtin_amdgcn_smfmac_f32_32x32x64_bf8_bf8(a, b, c, idx, 0, 0);
  }
};

template <> struct mma32<i8_t> {
  using acc_t = int16v;
  using acc4_t = int4v;
  static __device__ __forceinline__ int16v run(int4v a, int8v b, int16v c, int idx) {
    return __builtin_amdgcn_smfmac_i32_32x32x64_i8(a, b, c, idx, 0, 0);
  }
};

template <int WAVES_J_, int TJ_, int TI_ = 4, int RING_ = 3>
struct TileCfgT {
  static constexpr int WAVES_I = 2, WAVES_J = WAVES_J_;
  static constexpr int NW = WAVES_I * WAVES_J;
  static constexpr int THREADS = 64 * NW;
  static constexpr int TI = TI_, TJ = TJ_;       // 32x32 instructions per wave
  static constexpr int WI = 32 * TI, WJ = 32 * TJ;
  static constexpr int BI = WI * WAVES_I, BJ = WJ * WAVES_J;
  static constexpr int RING = RING_;             // stage buffers
  static_assert((BI == 128 && BJ == 64) || ((BI == 128 || BI == 192) && BJ == 128) || (BI == 256 && (BJ == 256 || BJ == 192 || BJ == 128 || BJ == 64)) || (BJ == 192 && (BI == 192 || BI == 384)),
                "stage buffers are sized for 256-row tiles of 256, 192, 128 or 64 columns, 192-column tiles of 192 or 384 rows, 128-column tiles of 128 or 192 and 64-column tiles of 128");
  static constexpr int KB = 128;                 // bytes of dense k per row per stage
  static constexpr int STEPS = KB / 64;          // instruction steps per stage
  static constexpr int A_ROW = KB / 2;           // LDS bytes per row per stage: compressed values
  static constexpr int B_ROW = KB;               //                              dense operand
  static constexpr int GH = BI == 384 ? 6 : 8;   // raster group height in tiles along i
  static constexpr int NB = BJ * B_ROW / 1024 / NW;   // 1 KB copies per wave per stage: B
  static constexpr int NA = BI * A_ROW / 1024 / NW;   //                                 A values
};
using TiledCfg = TileCfgT<4, 2>;
// The same 256 x 256 tile on four waves, one per SIMD, each computing 128 x 128 with 256 accumulator registers
// (the 512-register budget of a wave that has its SIMD to itself).  Every fragment read from LDS then feeds four
// matrix instructions instead of two or four: 100 KB of fragment reads per stage instead of 132 KB.  In cycles the
// two forms are equal (the matrix pipes are busy for 0.72 of them on config 3 either way), but the kernel runs
// against the power limit, and with 29 % fewer LDS cycles the clock settles higher: 0.5 to 2.7 % less time on the
// fp16 products of 8192 x 4096 x 11008 (more on boxes with less power headroom), 2.8 to 4.6 % on the fp8 product of
// 16384 x 8192 x 8192.  With few stages per tile the longer prologue and output pass of a
// 4-wave workgroup cost more than that (12 stages: 8 % slower; 24: equal; 32: 0.6 to 1.3 % faster), so only chained
// tiles of kWave4MinStages or more stages take this form (256 x 192 and 384 x 192 tiles: choose_short).
using Wave4Cfg = TileCfgT<2, 4>;
// 256 x 192 tiles in the 4-wave form (wave tile 128 x 96): a tile costs 0.89 of a 256 x 256 one, so where the
// narrower tiles need no more rounds of the compute units than the wide ones, every round is that much shorter
// (W[1600, 6400] against 12288 tokens: 336 wide tiles or 448 narrow ones, two rounds either way, 147 against 165 us;
// W[11008, 4096] against 2048 tokens alike).  Below kWave4MinStages stages choose_short decides.
using Wave4Cfg192 = TileCfgT<2, 3>;
// 192 x 192 tiles in the 4-wave form (wave tile 96 x 96, 144 accumulators): where rounds of the compute units fill better with
// them (takes_square).  A stage takes 0.53 us against 0.93 of a 256 x 256 one for 0.5625 of its work, but 0.67 against 1.0 at the
// clock that full rounds sustain.  With a quarter of the accumulators free they also hold the transposing fragment reads of a
// k-strided dense operand, which the other two 4-wave tiles spill.  us, 256 rows a tile and now, fp16: 6400 x 1600 against 2800
// columns 53.3 -> 38.5, 768 x 3072 against 12288 43.5 -> 42.0 (bound by the 75 MB of its dense operand: 34 where they come from the
// last cache); e4m3 5760 x 2688 against 6023 75.5 -> 62.1; k-strided 3072 x 12288 against 768 columns 50.8 -> 44.2, 768 x 12288
// against 3072 57.4 -> 51.4, 3072 x 1024 against 768 16.6 -> 13.1 (40 products of 8 to 253 stages: 14 % less on average).
// Two stage buffers and two workgroups to a compute unit (76 KB and 256 registers each) instead of three buffers and
// chained tiles: 36.2 and 35.9 us for the first, 52.0 and 41.8 for the second.
using SquareCfg = TileCfgT<2, 3, 3>;
// 384 x 192 tiles in the 4-wave form (wave tile 192 x 96, 288 accumulators; 16-bit operands: the stage buffers of 8-bit ones do
// not fit): 1.125 of the work of a 256 x 256 tile, for products whose tiles of the other sizes leave much of their last round of the
// compute units empty (takes_tall).  At equally full rounds it takes what 256 x 256 tiles take (8192 x 8192 against 8192 columns,
// four rounds of either, 518 and 497 us).  us on the other tiles and on these, fp16: 11008 x 4096 against 8192 columns 358 -> 346
// (5.4 rounds -> 4.9), 6144 x 12288 against 3000 251 -> 205 (three rounds of 192 x 192 tiles -> one), 6144 x 8192 against 6144
// 320 -> 280, 6144 x 3072 against 3000 64.9 -> 57.0, 1536 x 4096 against 12288 98 -> 77.  Raster groups of 5, 6 and 8 tiles: 346, 348
// and 349 us for the first product, 342, 342 and 346 for 10752 x 4096 against 8192.  All vector registers are kept; 51 to 60 scalar ones
// are spilled (35 to 46 in the other 4-wave forms), none of them inside the stage loop.
using TallCfg = TileCfgT<2, 3, 6>;
constexpr int kWave4MinStages = 32;
constexpr int kRotateMinStages = 56;
static_assert(kRotateMinStages - 2 - (7 * kRotateMinStages >> 3) >= 1, "the first three stages of a tile are copied before the order wraps");
// 128 x 64 tiles, four waves (wave tile 64 x 32, 32 accumulators), four stage buffers: for dense operands of at most 64 columns (a few dozen
// tokens), where a wider tile would copy and multiply clamped columns.  17 KB per stage, two blocks per CU.  These products are short: the pass
// over the compressed operand takes a few us, and the rest is the launch, the first stage's way from memory, one stage after the other and the sum of the
// pieces.  us on 256 x 64 tiles of two waves with three buffers, on these of two waves, of four, each with its best number of pieces:
// fp16 4096 x 4096 against 64 columns 13.5, 12.1, 11.1; 8192 x 8192 against 64 23.1, 21.1, 20.8; 4096 x 11008 against 40 18.9, 16.2, 15.7;
// 5120 x 1280 against 64 11.9, 8.9, 7.2; e4m3 4096 x 4096 against 64 11.5, 10.4, 9.6.  Of 100 products of 128 to 20480 rows, 2 to
// 512 stages and 8 to 64 columns 97 are faster, 17 % on average over all (3840 x 1280 against 8 columns would be 4.8 and 5.2, but takes spmm_few); of weights of
// 85 to 98 rows of tiles some are slower, whose two pieces fill the units less well than four or five of half as many did: 11072 x 12352 against 56 38.6 and 40.2.
using SlimCfg = TileCfgT<2, 1, 2, 4>;
// 256 x 64 tiles, two waves, three stage buffers: the same for tall weights (takes_tall_slim)
using TallSlimCfg = TileCfgT<1, 2>;
// 256 x 128 tiles, four waves: products that these cover in one round of the compute units and the smaller tiles below do not (takes_mid)
using MidCfg = TileCfgT<2, 2>;
// 128 x 128 tiles, four waves (wave tile 64 x 64, 64 accumulators), where there is at most one for each compute unit (takes_small).  A product
// of one round takes as long as its tile: prologue, stages one after the other, output pass.  Here that is 4.6 us and 0.21 to 0.3 a stage, against 5.6 and
// 0.33 with 256 x 128 tiles, and with k in pieces a tile has half the partial sums to write.  What bounds it: a stage
// moves 25 KB into LDS and 48 KB out of it to the registers for 0.12 us of matrix instructions.  Four stage buffers instead of three (a
// stage is that much shorter, and its copies take no less time to arrive): us with 3, 4, 5 and 6 of them 3072 x 768 against
// 952 columns 7.9, 7.6, 7.9, 8.1; 1824 x 2048 against 704 13.1, 11.8, 12.2, 12.4; 6144 x 4096 against 424 24.6, 21.5, -, 21.9.
using SmallCfg = TileCfgT<2, 2, 2, 4>;
// 192 x 128 tiles, four waves (wave tile 96 x 64), four stage buffers: products that these cover in one round of the compute units and 128 x 128
// tiles do not (takes_lower)
using LowerCfg = TileCfgT<2, 2, 3, 4>;

// ACTS: the kernel is built twice, for launches without an activation (output pass: plain or bias only) and with one
// (bias or zeros, then ReLU, SiLU or GELU); with all five passes in one kernel the compiler no longer keeps the
// wave-uniform copy addresses in scalar registers.
template <typename T, typename OutT, bool C_JMAJOR, typename C, bool B_KSTRIDED, bool PERSIST, bool ACTS = false>
__global__ void __launch_bounds__(C::THREADS)
spmm_pipe(const uint8_t* __restrict__ a_values, const uint8_t* __restrict__ a_meta, int64_t n_sparse, int64_t k,
          const uint8_t* __restrict__ b, int64_t ldb_bytes, int64_t n_dense,
          OutT* __restrict__ c, int64_t ldc, const OutT* __restrict__ bias, float scale, int act,
          int tiles_i, int tiles_j, int splits, float* __restrict__ partial, int aux) {
  constexpr int ES = sizeof(T);
  constexpr int M_ROW = ES == 2 ? C::KB / 16 : C::KB / 8;   // metadata bytes per row per stage (8 or 16)
  constexpr int M_STEP = M_ROW / C::STEPS;
  // Metadata: in the panel form the words of 32 dense columns of consecutive rows are adjacent, [k/32][m][4 B],
  // so the 256 rows of a tile are one 1 KB run per block of 32 columns and a stage is M_ROW/4 such runs (2 for
  // 16-bit values, 4 for 8-bit ones).  In LDS they lie in the same order, [block][row][4 B], which is the order
  // the index operands are read in: 16-bit values read the halfword of their k half from block = step; 8-bit
  // values the dword of block = 2*step + k half; consecutive lanes read consecutive words either way.
  // A run is one 16-byte-per-lane copy instruction; 8-bit values take those, issued by the last waves of the
  // workgroup (copied a dword per lane, 16 instructions per stage, the same bytes took a fifth of the fp8
  // kernel's copy time).  With 16-bit values and more waves than runs every wave brings a quarter run (or more)
  // with dword copies instead, so that all waves run the same code: a branch in the loop body makes the compiler
  // re-mask the 16-bit index words behind it, and that wait for all of a step's reads costs 5 %.  (Runs of 192 rows
  // are three quarters; where those do not divide among the waves, the last ones are copied twice, with the same bytes.)
  constexpr int STAGE_KB = M_ROW / 4;                        // 1 KB metadata runs per stage
  constexpr bool M_DWORD = (ES == 2 && C::NW > STAGE_KB) || C::BI != 256;   // quarter runs, every wave
  constexpr int MWAVES = M_DWORD ? C::NW : (STAGE_KB < C::NW ? STAGE_KB : C::NW);   // waves that copy metadata
  constexpr int QUARTERS = C::BI / 64;                       // of a run
  constexpr int MCOPIES = M_DWORD ? STAGE_KB * QUARTERS : STAGE_KB;
  constexpr int MW = (MCOPIES + MWAVES - 1) / MWAVES;        // copies per such wave
  static_assert(MW * MWAVES == MCOPIES || C::BI != 256, "metadata copies must divide among the waves");
  static_assert(M_DWORD || C::BI == 256, "full runs are 256 rows");
  constexpr bool M_HALF_MAJOR = ES == 1;
  // one stage buffer = [A values | B | A metadata]; C::RING (three or four) of them rotate
  constexpr int A_STAGE = C::BI * C::A_ROW, B_STAGE = C::BJ * C::B_ROW, M_STAGE = C::BI * M_ROW;
  constexpr int B_AT = A_STAGE, M_AT = A_STAGE + B_STAGE, STAGE_BYTES = A_STAGE + B_STAGE + M_STAGE;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[C::RING * STAGE_BYTES];

  // ---- XCD-aware work assignment.  A unit of work is (k-split, tile); units are ordered split-major
  // so that the units resident on an XCD belong to the same k range and share operand rows in L2.
  // Workgroup ids are dealt to the 8 XCDs round-robin: XCD x owns the units [x * per_xcd, (x+1) * per_xcd),
  // its workgroup number s = id / 8 takes unit s of that range -- and, PERSIST, every `slots`-th one after
  // it (slots = workgroups per XCD), one tile after the other in the same pipeline.
  const int ntiles = tiles_i * tiles_j;
  const int nunits = ntiles * splits;
  const int per_xcd = (nunits + 7) / 8;
  const int bid = blockIdx.x;
  const int slots = PERSIST ? (int)(gridDim.x >> 3) : per_xcd;
  const int xcd_end = min(((bid & 7) + 1) * per_xcd, nunits);
  int unit = (bid & 7) * per_xcd + (bid >> 3);
  if (unit >= xcd_end) return;
  constexpr int GH = C::GH;
  // aux: chained tiles (PERSIST) -- the start stagger in 10 ns ticks; otherwise the first row of tiles of this launch
  // (a launch may cover the tile rows [aux, aux + tiles_i) of the product; n_sparse stays the row count of the whole operand)
  const int stagger_ticks = PERSIST ? aux : 0;
  const int tile_row0 = PERSIST ? 0 : aux;
  int64_t i0 = 0, j0 = 0;
  const int split = PERSIST ? 0 : __builtin_amdgcn_readfirstlane(unit / ntiles);                // k piece
  int group = __builtin_amdgcn_readfirstlane((unit - split * ntiles) / (GH * tiles_j)), in_group = unit - split * ntiles - group * (GH * tiles_j);
  // origin of the tile number in_group of the group: the divisor is GH but for the last group (a division by a number that is not
  // known to the compiler is some 40 instructions, which nothing covers where one wave has a SIMD)
  auto locate = [&](int64_t& ti0, int64_t& tj0) {
    const int gh = min(GH, tiles_i - group * GH);
    int col = (unsigned)in_group / GH;
    if (gh != GH) col = __builtin_amdgcn_readfirstlane((unsigned)in_group / (unsigned)gh);
    ti0 = (int64_t)(tile_row0 + group * GH + (in_group - col * gh)) * C::BI;
    tj0 = (int64_t)col * C::BJ;
  };
  auto advance = [&]() {                                       // to the workgroup's next tile
    in_group += slots;
    for (int size = min(GH, tiles_i - group * GH) * tiles_j; in_group >= size; size = min(GH, tiles_i - group * GH) * tiles_j) {
      in_group -= size;
      group++;
    }
  };
  locate(i0, j0);
  // Chained tiles: every second workgroup of an XCD starts `stagger_ticks` (10 ns each) late.  All compute units
  // otherwise finish their tiles at the same moment and write them out together, at the HBM rate, while no matrix
  // instruction issues (a wave's stores share the counter its copies are waited on, so the next tile stalls until
  // they are acknowledged); with two groups half a burst apart each group's stores drain while the other
  // multiplies.
  if constexpr (PERSIST) {
    if (stagger_ticks > 0 && ((bid >> 3) & 1)) {
      const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
      for (int spin = 0; spin < 1024 && __builtin_amdgcn_s_memrealtime() - t0 < (uint64_t)stagger_ticks; spin++)
        __builtin_amdgcn_s_sleep(4);                 // (also bounded in iterations, whatever the counter does)
    }
  }

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wi = wave / C::WAVES_J, wj = wave % C::WAVES_J;
  const int l32 = lane & 31, lh = lane >> 5;
  const int nstages_total = (int)((k * ES) / C::KB);
  const int st_begin = (int)((int64_t)split * nstages_total / splits);
  const int nstages = (int)((int64_t)(split + 1) * nstages_total / splits) - st_begin;
  // The tiles of XCD x take their stages from the x-th eighth of k on and wrap round (4-wave form, kRotateMinStages or more).
  // A stage of the dense operand is 128 bytes from each of 256 rows, whose pitch is often a multiple of some
  // 4 KB: with all XCDs at the same stage the whole chip reads the same few memory channels at a time, and the copies, two
  // stages ahead, arrive late wherever the operand comes from memory and not from the last cache.  What counts is stages and
  // not elements.  us on operands that change from product to product, without and with: 24 to 32 stages alike; 40 and 48
  // within 0.7 % but for some products on square tiles (e4m3 3040 x 5120 against 6130 columns 69.7 -> 61.9); 56 e4m3 8192 x 7168
  // against 8192 233 -> 227, 3040 x 7168 against 6130 84.4 -> 80.7, fp16 5120 x 3584 against 5000 112.2 -> 112.7; 64 fp16
  // 4096 x 4096 against 3001 56.5 -> 53.8, 11008 x 4096 against 8192 358.1 -> 358.4, e4m3 8192 x 8192 against 16384 541.9 -> 513.7;
  // 128 fp16 8192 x 8192 against 8192 530 -> 504; 172 bf16 4096 x 11008 against 3001 144.1 -> 132.9.  On the same operands 60 products
  // of 40 to 128 stages are within 0.4 %.  By halves or quarters of k instead of eighths 134 and 133 for the last, three stages
  // apart 138.  (So two equal rows of the dense operand may differ in the last bits of their sums where their tiles are on two XCDs;
  // the same call gives the same bits.)
  constexpr bool ROTATE = PERSIST && C::NW == 4;
  const int rot = ROTATE && nstages >= kRotateMinStages ? (bid & 7) * nstages >> 3 : 0;
  const int st_first = st_begin + rot;

  // ---- per-lane global sources of the copies (first stage of this unit); LDS destinations are wave-uniform.
  // B: copy q of a wave brings 8 rows x 128 bytes; lane -> (row, swizzled chunk).
  // A: stage st of rows i0..i0+255 is one contiguous run of 256*64 value bytes at (st*n_sparse + i0)*64
  //    (and 256*M_ROW metadata bytes): copy q brings 16 rows x 64 bytes.
  // Every source is (tile base, uniform, advanced by whole stages) + (lane offset inside the tile's first stage).
  uint32_t ob[C::NB], oa[C::NA], om[MW];
  auto m_copy = [&](int q) {                     // which of the stage's metadata copies is the q-th of this wave
    const int c = (wave - (C::NW - MWAVES)) * MW + q;
    return MW * MWAVES == MCOPIES ? c : min(c, MCOPIES - 1);
  };
  const uint8_t *tile_b, *tile_a, *tile_m;
  // B with k strided (element (k,j) at k*ldb + j, 16-bit types): the stage is kept as [64 k][BJ j]
  // in LDS, copy q brings 1 KB of it (2 k-rows of 256 columns); 16-byte chunks are XOR-swizzled with
  // ((k & 3) << 1) | ((k >> 3 & 1) << 3) so that the transposing fragment reads below (four k-rows x
  // 32 bytes per 16 lanes) touch every bank once.  Rows of 192 columns start half of the banks apart by
  // themselves, and their 24 chunks go with ((k >> 1 & 1) << 2) | ((k >> 3 & 1) << 1).
  // Columns past n_dense re-read the last chunk.
  auto kstrided_swizzle = [](int krow) {
    return C::BJ == 256 ? ((krow & 3) << 1) | (((krow >> 3) & 1) << 3) : (((krow >> 1) & 1) << 2) | (((krow >> 3) & 1) << 1);
  };
  constexpr int64_t B_STAGE_ADVANCE_ROWS = B_KSTRIDED ? C::KB / ES : 0;
  const int64_t b_stage_stride = B_KSTRIDED ? B_STAGE_ADVANCE_ROWS * ldb_bytes : (int64_t)C::B_ROW;
  bool lanes_whole = false;
  auto point_at = [&](int64_t ti0, int64_t tj0) {              // sources of the first stage of the tile at (ti0, tj0)
    // (PERSIST: the lane id is made opaque here and in the output pass, so that the per-lane terms of the
    // addresses are formed again for every tile instead of living in registers through the main loop,
    // where the accumulators and two fragment sets leave none to spare)
    int lane = threadIdx.x & 63;
    if constexpr (PERSIST) asm volatile("" : "+v"(lane));
    const int64_t last_j = n_dense - 1 - tj0, last_i = n_sparse - 1 - ti0;       // >= 0: tile origins lie inside
    if constexpr (B_KSTRIDED) tile_b = b + (int64_t)st_first * B_STAGE_ADVANCE_ROWS * ldb_bytes;   // columns stay absolute: the clamp may step left of the tile
    else tile_b = b + tj0 * ldb_bytes + (int64_t)st_first * C::B_ROW;
    tile_a = a_values + (ti0 + (int64_t)st_first * n_sparse) * 64;
    tile_m = a_meta + (ti0 + (int64_t)st_first * STAGE_KB * n_sparse) * 4;
    // the lanes' offsets are those of any other tile unless rows of one of the two are clamped
    const bool whole = !B_KSTRIDED && last_j >= C::BJ - 1 && last_i >= C::BI - 1;
    if (whole && lanes_whole) return;
    lanes_whole = whole;
#pragma unroll
    for (int q = 0; q < C::NB; q++) {
      if constexpr (B_KSTRIDED) {
        constexpr int CHUNKS = C::BJ / 8;        // of a k-row
        const int piece = (wave * C::NB + q) * 64 + lane, krow = piece / CHUNKS;
        const int ch = (piece % CHUNKS) ^ kstrided_swizzle(krow);
        const int64_t col = min(tj0 + ch * 8, n_dense - 8);
        ob[q] = (uint32_t)(krow * ldb_bytes + col * ES);
      } else {
        const int row = (wave * C::NB + q) * 8 + (lane >> 3);
        const int ch = (lane & 7) ^ ((row >> 1) & 7);
        ob[q] = (uint32_t)(min((int64_t)row, last_j) * ldb_bytes + ch * 16);
      }
    }
#pragma unroll
    for (int q = 0; q < C::NA; q++) {
      const int row = (wave * C::NA + q) * 16 + (lane >> 2);
      const int ch = (lane & 3) ^ ((row >> 2) & 3);
      oa[q] = (uint32_t)(min((int64_t)row, last_i) * 64 + ch * 16);
    }
#pragma unroll
    for (int q = 0; q < MW; q++) {
      const int c = m_copy(q);                                 // quarter run (a lane brings one row's word) or run (4 rows' words)
      om[q] = M_DWORD ? (uint32_t)(((c / QUARTERS) * n_sparse + min((int64_t)((c % QUARTERS) * 64 + lane), last_i)) * 4)
                      : (uint32_t)((c * n_sparse + min((int64_t)lane * 4, last_i - 3)) * 4);
    }
  };
  point_at(i0, j0);
  const int64_t a_stage_stride = n_sparse * 64, m_stage_stride = n_sparse * M_ROW;
  constexpr int NCOPY = C::NB + C::NA + MW;      // copies per wave per stage (MW fewer for the waves without metadata)
  const bool has_meta = MWAVES == C::NW || wave >= C::NW - MWAVES;      // the last waves (measured: 2.7 % better than the first ones at fp8)

  // copy q of this wave for stage st into the stage buffer at LDS byte address `dst`
  const uint32_t smem_at = lds_offset(smem);
  auto issue_one = [&](int q, uint32_t dst) {
    if (q < C::NB) g2l16(tile_b, ob[q], dst + B_AT + (wave * C::NB + q) * 1024);
    else if (q < C::NB + C::NA) g2l16(tile_a, oa[q - C::NB], dst + (wave * C::NA + q - C::NB) * 1024);
    else if constexpr (M_DWORD) g2l4(tile_m, om[q - C::NB - C::NA], dst + M_AT + m_copy(q - C::NB - C::NA) * 256);
    else if (has_meta) g2l16(tile_m, om[q - C::NB - C::NA], dst + M_AT + m_copy(q - C::NB - C::NA) * 1024);
  };
  // the sources advance a stage behind each stage's copies (formed from a stage number they cost four more scalar instructions)
  auto next_stage = [&]() { tile_b += b_stage_stride; tile_a += a_stage_stride; tile_m += m_stage_stride; };
  auto issue = [&](uint32_t dst) {
#pragma unroll
    for (int q = 0; q < NCOPY; q++) issue_one(q, dst);
    next_stage();
  };

  typename mma32<T>::acc_t acc[C::TI][C::TJ];
#pragma unroll
  for (int ti = 0; ti < C::TI; ti++)
#pragma unroll
    for (int tj = 0; tj < C::TJ; tj++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[ti][tj][r] = 0;

  // ---- fragment offsets (swizzled)
  const int a_row = wi * C::WI + l32, b_row = wj * C::WJ + l32;
  const int a_sw = (l32 >> 2) & 3, b_sw = (l32 >> 1) & 7;
  int a_off[C::STEPS], b_off[C::STEPS][2];
#pragma unroll
  for (int step = 0; step < C::STEPS; step++) {
    a_off[step] = a_row * C::A_ROW + (((step * 2 + lh) ^ a_sw) * 16);
#pragma unroll
    for (int h = 0; h < 2; h++) b_off[step][h] = b_row * C::B_ROW + (((step * 4 + h * 2 + lh) ^ b_sw) * 16);
  }
  const int m_off = M_HALF_MAJOR ? lh * (C::BI * 4) + a_row * 4 : a_row * M_STEP + lh * (M_STEP / 2);   // inside a step's block
  constexpr int M_FRAG = M_HALF_MAJOR ? 32 * 4 : 32 * M_STEP;    // from one 32-row fragment to the next
  // k-strided B: transposing reads (DS_READ_B64_TR_B16).  In a group of 16 lanes, lane i receives
  // the halfwords i%4 of the source lanes 4e + i/4 (e = 0..3).  Source lane s therefore addresses
  // k-row k0 + s/4, halfwords 4*(s%4).. of the group's 16 columns, and lane i ends up with
  // k0..k0+3 of column i: four such reads (k0 = 8*kb + {0, 4, 16, 20}) make one dense fragment.
  int bt_off[C::TJ];
  if constexpr (B_KSTRIDED) {
    const int g16 = lane >> 4, s16 = lane & 15;
    const int kb = g16 >> 1, jbase = (g16 & 1) * 16;
    const int swz = kstrided_swizzle(kb * 8 + (s16 >> 2));        // the same for all four rows read
#pragma unroll
    for (int tj = 0; tj < C::TJ; tj++) {
      const int col = wj * C::WJ + tj * 32 + jbase + (s16 & 3) * 4;  // halfword column in the tile
      bt_off[tj] = (kb * 8 + (s16 >> 2)) * (C::BJ * 2) + (((col >> 3) ^ swz) * 16) + ((col >> 2) & 1) * 8;
    }
  }

  // ---- main loop: a software pipeline over instruction steps.  While the matrix instructions of a
  // step run from one register set, the fragments of the next step are read from LDS into the
  // other, a few reads after every row of instructions: read in a block at the start of a step, the
  // eight waves' requests fill the LDS queue, every wave stalls on issue, and the matrix pipes wait.
  // The copies of the stage two ahead are spread over the same gaps (issued in a burst they would
  // queue in the texture-address unit and hold back the fragment reads).
  // One workgroup barrier per stage, B(s), placed before the first fragment read of stage s: every
  // wave arrives having waited for its own copies of stage s and with all its reads of stage s-1
  // complete, so behind B(s) stage s is visible and the buffer of stage s-1 is free for the copies
  // of stage s+2.  The matrix instructions of the last step of stage s-1 are issued behind B(s),
  // from registers, with the first reads of stage s between them.
  int4v af[2][C::TI];
  int idx[2][C::TI];
  int4v bf[2][C::TJ][2];                         // the two 16-byte halves of a dense fragment
  short4v bq[2][C::TJ][4];                       // k-strided B: the four 8-byte quarters
  // The reads of a step, in the order the next step's instructions need them: its first row of
  // instructions takes every dense fragment and sparse fragment 0, row r then only needs sparse
  // fragment r.  Read n: dense half-fragment n (fragment n/2, half n%2) for n < 2*TJ, then sparse
  // fragment and index word alternately.
  constexpr int B_READS = (B_KSTRIDED ? 4 : 2) * C::TJ;
  constexpr int N_READS = B_READS + 2 * C::TI;
  constexpr int READS_PER_ROW = (N_READS + C::TI - 1) / C::TI;
  // `src` is the byte offset of the stage buffer in smem (wave-uniform, changes every stage): the
  // per-lane addresses are formed when needed and fragment offsets ride in the instructions' immediates
  auto read_one = [&](int set, int n, uint32_t src, int step) {
    const uint8_t* base = smem + src;
    if (n < B_READS) {
      if constexpr (B_KSTRIDED) {
        const int tj = n >> 2, quarter = n & 3;                  // quarter: k0 = 8*kb + {0, 4, 16, 20}
        const uint8_t* src_q = base + B_AT + bt_off[tj] + step * (32 * C::BJ * 2) + ((quarter & 1) * 4 + (quarter >> 1) * 16) * (C::BJ * 2);
        bq[set][tj][quarter] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(lds_ptr_t)src_q);
      } else {
        bf[set][n >> 1][n & 1] = *reinterpret_cast<const int4v*>(base + B_AT + b_off[step][n & 1] + (n >> 1) * 32 * C::B_ROW);
      }
    } else {
      const int f = (n - B_READS) >> 1;
      if (((n - B_READS) & 1) == 0) af[set][f] = *reinterpret_cast<const int4v*>(base + a_off[step] + f * 32 * C::A_ROW);
      else if constexpr (ES == 2) idx[set][f] = *reinterpret_cast<const uint16_t*>(base + M_AT + m_off + f * M_FRAG + step * (C::BI * M_STEP));
      else idx[set][f] = *reinterpret_cast<const int*>(base + M_AT + m_off + f * M_FRAG + step * (C::BI * M_STEP));
    }
  };
  // `half` selects which half of the wave's copies of stage pst is issued between the instructions
  // (into the buffer at LDS address dst); with `reads`, the fragments of step rstep of the buffer at
  // offset src go into the other register set.
  constexpr int PER_SLOT = (NCOPY + 2 * C::TI - 1) / (2 * C::TI);
  // copies of a stage issued during the first of its two steps (the rest during the second)
  constexpr int FIRST_HALF_COPIES = C::NW == 4 ? (NCOPY + 1) / 2 : (C::TI * PER_SLOT < NCOPY ? C::TI * PER_SLOT : NCOPY);
  auto dense_fragment = [&](int set, int tj) {
    if constexpr (B_KSTRIDED) {
      typedef int int2v __attribute__((ext_vector_type(2)));
      const int2v q0 = __builtin_bit_cast(int2v, bq[set][tj][0]), q1 = __builtin_bit_cast(int2v, bq[set][tj][1]);
      const int2v q2 = __builtin_bit_cast(int2v, bq[set][tj][2]), q3 = __builtin_bit_cast(int2v, bq[set][tj][3]);
      return int8v{q0[0], q0[1], q1[0], q1[1], q2[0], q2[1], q3[0], q3[1]};
    } else {
      const int4v lo = bf[set][tj][0], hi = bf[set][tj][1];
      return int8v{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
  };
  auto mma_step = [&](int set, int half, bool copies, uint32_t dst, bool reads, uint32_t src, int rstep) {
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (C::NW == 4) {
      // One wave per SIMD: no other wave fills the matrix pipe while this one issues reads and copies, so they go
      // one by one behind every matrix instruction instead of in a block behind a row of them (in blocks: 5 % slower
      // than the 8-wave form instead of faster).  Ending the reads a few instructions before the step does, so
      // that the stage barrier finds them landed, changes nothing measurable.
      constexpr int SLOTS = C::TI * C::TJ;
      static_assert(!B_KSTRIDED || C::TI * C::TJ <= 9, "with the transposing reads of a k-strided dense operand wave tiles of 128 x 128 spill");
#pragma unroll
      for (int ti = 0; ti < C::TI; ti++) {
#pragma unroll
        for (int tj = 0; tj < C::TJ; tj++) {
          acc[ti][tj] = mma32<T>::run(af[set][ti], dense_fragment(set, tj), acc[ti][tj], idx[set][ti]);
          __builtin_amdgcn_sched_barrier(0);
          const int n = ti * C::TJ + tj;
          if (reads) {
#pragma unroll
            for (int u = 0; u < (N_READS + SLOTS - 1) / SLOTS; u++)
              if (n * N_READS / SLOTS + u < (n + 1) * N_READS / SLOTS) read_one(set ^ 1, n * N_READS / SLOTS + u, src, rstep);
          }
#pragma unroll
          for (int q = 0; q < NCOPY; q++)
            if ((q * 2 * SLOTS) / NCOPY == half * SLOTS + n && copies) issue_one(q, dst);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      return;
    }
#pragma unroll
    for (int ti = 0; ti < C::TI; ti++) {
#pragma unroll
      for (int tj = 0; tj < C::TJ; tj++) {
        acc[ti][tj] = mma32<T>::run(af[set][ti], dense_fragment(set, tj), acc[ti][tj], idx[set][ti]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (reads) {
#pragma unroll
        for (int u = 0; u < READS_PER_ROW; u++)
          if (ti * READS_PER_ROW + u < N_READS) read_one(set ^ 1, ti * READS_PER_ROW + u, src, rstep);
      }
#pragma unroll
      for (int u = 0; u < PER_SLOT; u++) {
        const int q = (half * C::TI + ti) * PER_SLOT + u;
        if (q < NCOPY && copies) issue_one(q, dst);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  static_assert(C::STEPS == 2, "the pipeline below is written for two instruction steps per stage");
  static_assert(!PERSIST || C_JMAJOR, "chained tiles rely on the wait inside the j-major output passes");
  constexpr int LEAD = C::RING - 1;              // stages that the copies run ahead
  static_assert(LEAD == 2 || (!PERSIST && MWAVES == C::NW), "longer rings: tiles that are not chained, the same copies in every wave");
  auto stage_barrier = [&](bool more) {          // B(st+1): only this wave's copies of the stages from st+2 on may still fly
    if (!more) wait_copies_and_barrier<0, true>();
    else if (MWAVES == C::NW || has_meta) wait_copies_and_barrier<NCOPY * (LEAD - 1), true>();
    else wait_copies_and_barrier<NCOPY - MW, true>();
  };
  auto last_barrier = [&](int left) {            // the same where `left` stages follow st+1
    if constexpr (LEAD == 2) stage_barrier(left > 0);
    else if (left >= LEAD - 1) wait_copies_and_barrier<NCOPY * (LEAD - 1), true>();
    else if (LEAD > 4 && left == 3) wait_copies_and_barrier<NCOPY * 3, true>();
    else if (LEAD > 3 && left == 2) wait_copies_and_barrier<NCOPY * 2, true>();
    else if (left == 1) wait_copies_and_barrier<NCOPY, true>();
    else wait_copies_and_barrier<0, true>();
  };

  issue(smem_at);
#pragma unroll
  for (int ahead = 1; ahead < LEAD; ahead++)
    if (nstages > ahead) issue(smem_at + ahead * STAGE_BYTES);
  uint32_t cur = 0, nxt = STAGE_BYTES, fre = LEAD * STAGE_BYTES;   // buffers of stage st, st+1, st+LEAD (= st-1)
  auto turn = [&]() {                            // to the next stage's
    const uint32_t t = cur;
    cur = nxt;
    nxt = LEAD == 2 ? fre : nxt == LEAD * STAGE_BYTES ? 0 : nxt + STAGE_BYTES;
    fre = t;
  };
  // PERSIST (nstages >= 4, no k pieces): the workgroup walks its tiles in one pipeline.  The copies of
  // the next tile's first two stages are issued during the last two stages of the current one, into
  // the two buffers those stages leave free; the output pass then stages through the third (the last
  // stage's) while they fly, and the next tile starts with its operands already in LDS.
  int64_t next_i0 = 0, next_j0 = 0;
  bool has_next = false;
  bool chained = false;                          // this tile's first two stages were copied under the previous tile
  for (;;) {
  // A chained tile's first two stages were waited for by every wave before the first store of the previous
  // output pass (below), so its first two barriers only publish them: waiting here on the counter of
  // outstanding memory operations would wait for the acknowledgements of those stores, which it does not
  // tell from copies.  From the third barrier on the usual wait is enough again: stores may complete out of
  // order with loads, but loads complete in order, and after the copies of stage s a wave issues the NCOPY
  // copies of stage s + 1 before it waits -- if one copy of stage s were still in flight, all of those
  // would be too, more than the NCOPY operations the wait allows.
  if (PERSIST && chained) wait_reads_and_barrier();
  else last_barrier(nstages - 1);
  // stage 0: nothing to multiply yet
  {
    const bool more = PERSIST || LEAD < nstages;      // (chained tiles have four stages at least)
#pragma unroll
    for (int n = 0; n < N_READS; n++) read_one(0, n, cur, 0);
    if (more) {
#pragma unroll
      for (int q = 0; q < FIRST_HALF_COPIES; q++) issue_one(q, smem_at + fre);
    }
    mma_step(0, 1, more, smem_at + fre, true, cur, 1);
    if (more) next_stage();
    if (PERSIST && chained) wait_reads_and_barrier();
    else if (LEAD == 2) stage_barrier(more);
    else last_barrier(nstages - 2);
  }
  // stage st: behind B(st), register set 1 holds the last step of stage st-1
  int st = 1;
  // Up to the wrap of the stage order, to the last two stages, and, where a tile follows, through those: what they copy are its first two.
  // (Of one loop, and the next tile found with few instructions: nothing covers what a workgroup does between tiles, on four waves least
  // of all.  With two stages of their own, in which every copy stood behind a branch, and new lane offsets and four divisions for each
  // tile, us on operands that change, then and now: fp16 3072 x 768 against 12288 columns 44.8 and 43.0 on 8-wave tiles, 55 and 40 on
  // 256 x 192 ones; 2048 x 512 24.3 and 22.7; 6400 x 1600 against 6000 77.4 and 76.1; 11008 x 4096 against 8192 352.5 and 350.9.)
  has_next = false;
  for (int lim = nstages - LEAD - rot;;) {
    for (; st < lim; st++) {
      turn();
      mma_step(1, 0, true, smem_at + fre, true, cur, 0);
      mma_step(0, 1, true, smem_at + fre, true, cur, 1);
      next_stage();
      stage_barrier(true);
    }
    if (ROTATE && st < nstages - 2) {                // (lim >= 1: the wrap is behind the copies of stage 2)
      tile_b -= nstages * b_stage_stride;
      tile_a -= nstages * a_stage_stride;
      tile_m -= nstages * m_stage_stride;
      lim = nstages - 2;
      continue;
    }
    if (!PERSIST || st >= nstages || unit + slots >= xcd_end) break;
    unit += slots;                                   // every copy of this tile has been issued: aim at the next one
    has_next = true;
    advance();
    locate(next_i0, next_j0);
    point_at(next_i0, next_j0);
    lim = nstages;
  }
  for (; st < nstages; st++) {                       // the last LEAD stages of the last tile
    turn();
    mma_step(1, 0, false, 0, true, cur, 0);
    mma_step(0, 1, false, 0, true, cur, 1);
    if constexpr (LEAD == 2) stage_barrier(false);
    else last_barrier(nstages - 2 - st);
  }
  // ---- bias: every lane fetches the bias of WI/64 of its wave's rows here, one instruction step ahead of the
  // output pass, which hands them round the wave through LDS.  (Fetched per element inside the pass -- 128 two-byte
  // loads per lane, a wait behind every four -- the bias cost 2.8 us per 256 x 256 tile: 59 % on top of a 12-stage
  // tile, 31 % on a 64-stage one.)
  // The loaded bits are first touched behind that step (the empty asm statements): converted right away, the compiler
  // waits for each load -- and with it for every copy in flight -- before the step's matrix instructions.  They stand under no
  // condition: under a second test of the loads' own, the compiler sees a way to the next tile on which a load is never waited
  // for, and where its register is one of the stage loop's it waits there, in every stage, for every copy in flight (8-wave
  // tiles, fp16: W[6400, 1600] against 5000 columns 64.3 us that way, 56.9 this way, 6000 83.5 and 73.3, float32 results 93.8
  // and 85.7; k strided W[8192, 4096] against 8192 281 and 266).
  using accs_t = std::remove_reference_t<decltype(acc[0][0][0])>;
  constexpr int BIAS_Q = (C::WI + 63) / 64;
  const bool bias_f32 = sizeof(OutT) == 2 && (act & TF24_BIAS_F32);
  uint32_t bias_w[BIAS_Q];
#pragma unroll
  for (int q = 0; q < BIAS_Q; q++) bias_w[q] = 0;
  if (splits == 1 && bias != nullptr) {
#pragma unroll
    for (int q = 0; q < BIAS_Q; q++) {
      const int64_t row = i0 + wi * C::WI + q * 64 + (int)(threadIdx.x & 63);
      const int64_t at = row < n_sparse ? row : n_sparse - 1;
      if (bias_f32) bias_w[q] = reinterpret_cast<const uint32_t*>(bias)[at];      // (rounded where it is unpacked)
      else bias_w[q] = bias_bits(bias[at]);
    }
  }
  mma_step(1, 0, false, 0, false, 0, 0);       // the last step
#pragma unroll
  for (int q = 0; q < BIAS_Q; q++) asm volatile("" : "+v"(bias_w[q]));

  // ---- split-K: park the 32-bit accumulators in the workspace, in register order (every group of
  // four accumulators is one contiguous 16-byte-per-lane slab); spmm_reduce_splits finishes the job.
  if (splits > 1) {
    float* base = partial + (int64_t)unit * (C::BI * C::BJ);
#pragma unroll
    for (int ti = 0; ti < C::TI; ti++)
#pragma unroll
      for (int tj = 0; tj < C::TJ; tj++) {
        if (j0 + wj * C::WJ + tj * 32 >= n_dense) continue;      // columns past the dense operand: never read back
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const int slab = (ti * C::TJ + tj) * 4 + g;
          typename mma32<T>::acc4_t v = {acc[ti][tj][g * 4], acc[ti][tj][g * 4 + 1], acc[ti][tj][g * 4 + 2], acc[ti][tj][g * 4 + 3]};
          *reinterpret_cast<typename mma32<T>::acc4_t*>(base + ((int64_t)slab * C::THREADS + tid) * 4) = v;
        }
      }
    return;
  }

  // 16-bit j-major outputs leave in pieces of 32(j) x 32*PASS_TI(i): 64 i, or the whole 96 of a wave tile of three fragments
  // (rows of 192 bytes, 208 apart in LDS: 16 rows' chunks of one position lie on different banks)
  constexpr int PASS_TI = C::TI % 2 == 0 ? 2 : C::TI;
  constexpr int PITCH = PASS_TI == 2 ? 128 : PASS_TI * 64 + 16;
  constexpr int SLICE = 32 * PITCH;              // of the staging buffer, per wave
  static_assert(C::NW * (SLICE + BIAS_Q * 256) <= STAGE_BYTES, "the output pass stages through one stage buffer");
  auto output_pass = [&](auto mode_c) {
    constexpr int MODE = decltype(mode_c)::value;
    int lane = threadIdx.x & 63;
    if constexpr (PERSIST) asm volatile("" : "+v"(lane));
    const int l32 = lane & 31, lh = lane >> 5;
    // the bias of this wave's WI rows, behind the staging slices of all waves; the wave reads back what its own lanes
    // wrote (LDS accesses of one wave execute in order: no barrier)
    accs_t* bias_lds = reinterpret_cast<accs_t*>(smem + cur + C::NW * SLICE + wave * (BIAS_Q * 256));
    if constexpr (MODE != EPI_PLAIN) {
#pragma unroll
      for (int q = 0; q < BIAS_Q; q++) {
        uint32_t w = bias_w[q];
        if constexpr (sizeof(OutT) == 2)
          if (bias_f32) w = bias_bits(from_float<OutT>(__builtin_bit_cast(float, w)));
        const accs_t v = bias_as(accs_t(0), bias_from_bits<OutT>(w));
        bias_lds[q * 64 + lane] = i0 + wi * C::WI + q * 64 + lane < n_sparse ? v : accs_t(0);
      }
    }
    // The bias of rows ti*32 + g*8 + lh*4 + 0..3 of the wave's tile, g = 0..3: read for a whole block of the pass
    // ahead of its staging writes.  (Read where it is used, every quad waits behind the LDS writes issued before it,
    // 32 round trips per wave and tile: 1.3 to 2 us.)
    using bias4_t = typename mma32<T>::acc4_t;
    auto bias_quads = [&](int ti, bias4_t (&bq)[4]) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        bq[g] = bias4_t{0, 0, 0, 0};
        if constexpr (MODE != EPI_PLAIN) bq[g] = *reinterpret_cast<const bias4_t*>(bias_lds + ti * 32 + g * 8 + lh * 4);
      }
    };
    // ---- epilogue.  D layout: column l%32, rows 8*(r/4) + 4*(l/32) + r%4.
    // For 16-bit outputs stored j-major (the Y of X.W^T) a lane owns runs of only 4 consecutive i
    // (8 bytes) in 32 different output rows, so direct stores would touch 32 lines per instruction.
    // Instead every wave stages 32(j) x 64(i) pieces of its sub-tile in a private 4 KB slice of the
    // last stage's buffer (no wave reads it any more: the tile's last barrier is behind us; the other
    // two buffers may already be receiving the next tile) -- 128-byte rows, 16-byte chunks
    // XOR-swizzled with the row -- and streams them out as eight full 128-byte row segments per
    // instruction (streaming stores: the tile is not read again by this kernel and should not
    // displace operand lines in L2).  LDS accesses of one wave execute in order, so the passes need
    // no barrier between them.  (No wave_lds_fence either: with one around every piece 256 x 192 tiles take 13 accumulator
    // registers more, and 3072 x 768 against 12288 columns and 5120 x 1280 against 4416, of 12 and 20 stages, 1 to 3 % longer.)
    if constexpr (C_JMAJOR && sizeof(OutT) == 2) {
      uint8_t* stage = smem + cur + wave * SLICE;
      constexpr int CHUNKS = PASS_TI * 4;                       // 16-byte chunks of a row of the piece
      auto chunk_at = [](int row, int ch) { return row * PITCH + (PASS_TI == 2 ? ch ^ (row & 7) : ch) * 16; };
  #pragma unroll
      for (int tj = 0; tj < C::TJ; tj++) {
  #pragma unroll
        for (int ip = 0; ip < C::TI / PASS_TI; ip++) {          // 32 * PASS_TI sparse rows (i) per pass
          bias4_t bq[PASS_TI][4];
  #pragma unroll
          for (int t2 = 0; t2 < PASS_TI; t2++) bias_quads(ip * PASS_TI + t2, bq[t2]);
  #pragma unroll
          for (int t2 = 0; t2 < PASS_TI; t2++) {
            const int ti = ip * PASS_TI + t2;
  #pragma unroll
            for (int g = 0; g < 4; g++) {
              OutT o[4];
  #pragma unroll
              for (int r = 0; r < 4; r++) o[r] = to_out<OutT>(finish_element<MODE>(acc[ti][tj][g * 4 + r], scale, bq[t2][g][r]));
              *reinterpret_cast<Pack<OutT, 4>*>(stage + chunk_at(l32, t2 * 4 + g) + lh * 8) = *reinterpret_cast<Pack<OutT, 4>*>(o);
            }
          }
          // the next tile's first two stages (issued one and two stages ago) have to be in LDS before this
          // wave's first store joins the outstanding operations
          if (PERSIST && tj == 0 && ip == 0 && has_next) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  #pragma unroll
          for (int it = 0; it < CHUNKS / 2; it++) {
            // (in unsigned numbers: the corrections of signed divisions take registers, which the 8-wave kernels with an activation
            // then spill -- 18 of them, W[8192, 1024] fp16 with ReLU against 8192 columns 91 us instead of 84)
            const uint32_t piece = it * 64 + lane;
            const int jl = 64 % CHUNKS ? piece / CHUNKS : it * (64 / CHUNKS) + (uint32_t)lane / CHUNKS, ch = (64 % CHUNKS ? piece : (uint32_t)lane) % CHUNKS;
            const int64_t icol = i0 + wi * C::WI + ip * (32 * PASS_TI) + ch * 8;
            const int64_t jrow = j0 + wj * C::WJ + tj * 32 + jl;
            const int4v v = *reinterpret_cast<const int4v*>(stage + chunk_at(jl, ch));
            if (jrow < n_dense && icol < n_sparse) __builtin_nontemporal_store(v, reinterpret_cast<int4v*>(c + jrow * ldc + icol));
          }
        }
      }
    } else if constexpr (C_JMAJOR && sizeof(OutT) == 4) {
      // j-major 32-bit output (float32 from 8-bit operands, int32 from int8: the reference's output types for
      // them): the same staging with 32(j) x 32(i) pieces -- a lane's four consecutive i are one 16-byte chunk of
      // a 128-byte row -- so that the stores are full 128-byte row segments instead of 32-byte ones.
      uint8_t* stage = smem + cur + wave * SLICE;
      const int rr = lane >> 3, chr = lane & 7;
  #pragma unroll
      for (int tj = 0; tj < C::TJ; tj++) {
  #pragma unroll
        for (int ti = 0; ti < C::TI; ti++) {
          bias4_t bq[4];
          bias_quads(ti, bq);
  #pragma unroll
          for (int g = 0; g < 4; g++) {
            typedef OutT out4v __attribute__((ext_vector_type(4)));
            out4v o;
  #pragma unroll
            for (int r = 0; r < 4; r++) o[r] = to_out<OutT>(finish_element<MODE>(acc[ti][tj][g * 4 + r], scale, bq[g][r]));
            const int ch = g * 2 + lh;
            *reinterpret_cast<out4v*>(stage + l32 * 128 + ((ch ^ (l32 & 7)) * 16)) = o;
          }
          const int64_t icol = i0 + wi * C::WI + ti * 32 + chr * 4;
          // (chained tiles: see the 16-bit pass)
          if (PERSIST && tj == 0 && ti == 0 && has_next) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  #pragma unroll
          for (int it = 0; it < 4; it++) {
            const int jl = it * 8 + rr;
            const int64_t jrow = j0 + wj * C::WJ + tj * 32 + jl;
            const int4v v = *reinterpret_cast<const int4v*>(stage + jl * 128 + ((chr ^ (jl & 7)) * 16));
            if (jrow < n_dense && icol < n_sparse) __builtin_nontemporal_store(v, reinterpret_cast<int4v*>(c + jrow * ldc + icol));
          }
        }
      }
    } else if constexpr (!C_JMAJOR && sizeof(OutT) == 2 && C::TJ % 2 == 0) {
      // i-major 16-bit output (the W.B of `S @ dense`): a lane owns single elements of 64+ different
      // rows.  Stage 32(i) x 64(j) pieces as [i][64 j] (128-byte rows, chunks XOR-swizzled with the
      // row) and stream them out as eight full 128-byte rows per instruction.
      uint8_t* stage = smem + cur + wave * SLICE;
      const int rr = lane >> 3, chr = lane & 7;
  #pragma unroll
      for (int half = 0; half < C::TJ / 2; half++) {            // 64 output columns (j) per pass
  #pragma unroll
        for (int ti = 0; ti < C::TI; ti++) {                    // 32 sparse rows (i) per pass
          bias4_t bq[4];
          bias_quads(ti, bq);
  #pragma unroll
          for (int t2 = 0; t2 < 2; t2++) {
            const int tj = half * 2 + t2;
            const int jl = t2 * 32 + l32;
  #pragma unroll
            for (int g = 0; g < 4; g++) {
  #pragma unroll
              for (int r = 0; r < 4; r++) {
                const int il = g * 8 + lh * 4 + r;
                *reinterpret_cast<OutT*>(stage + il * 128 + (((jl >> 3) ^ (il & 7)) * 16) + (jl & 7) * 2) =
                    to_out<OutT>(finish_element<MODE>(acc[ti][tj][g * 4 + r], scale, bq[g][r]));
              }
            }
          }
          const int64_t jcol = j0 + wj * C::WJ + half * 64 + chr * 8;
  #pragma unroll
          for (int it = 0; it < 4; it++) {
            const int il = it * 8 + rr;
            const int64_t irow = i0 + wi * C::WI + ti * 32 + il;
            const int4v v = *reinterpret_cast<const int4v*>(stage + il * 128 + ((chr ^ (il & 7)) * 16));
            if (irow < n_sparse && jcol < n_dense) __builtin_nontemporal_store(v, reinterpret_cast<int4v*>(c + irow * ldc + jcol));
          }
        }
      }
    } else {
  #pragma unroll
      for (int ti = 0; ti < C::TI; ti++) {
        bias4_t bq[4];
        bias_quads(ti, bq);
  #pragma unroll
        for (int tj = 0; tj < C::TJ; tj++) {
          const int64_t col = j0 + wj * C::WJ + tj * 32 + l32;
  #pragma unroll
          for (int g = 0; g < 4; g++) {
            const int64_t row = i0 + wi * C::WI + ti * 32 + g * 8 + lh * 4;
            if (col >= n_dense || row >= n_sparse) continue;
            OutT o[4];
  #pragma unroll
            for (int r = 0; r < 4; r++) o[r] = to_out<OutT>(finish_element<MODE>(acc[ti][tj][g * 4 + r], scale, bq[g][r]));
            if constexpr (C_JMAJOR) {
              *reinterpret_cast<Pack<OutT, 4>*>(c + col * ldc + row) = *reinterpret_cast<Pack<OutT, 4>*>(o);
            } else {
  #pragma unroll
              for (int r = 0; r < 4; r++) c[(row + r) * ldc + col] = o[r];
            }
          }
        }
      }
    }
  };
  constexpr bool INT_ACC = std::is_same<typename mma32<T>::acc4_t, int4v>::value;
  if constexpr (!ACTS) {
    if (!bias) output_pass(std::integral_constant<int, EPI_PLAIN>{});
    else output_pass(std::integral_constant<int, EPI_BIAS>{});
  } else if constexpr (INT_ACC) {
    if ((act & ~TF24_BIAS_F32) == TF24_ACT_RELU) output_pass(std::integral_constant<int, EPI_RELU>{});
    else output_pass(std::integral_constant<int, EPI_BIAS>{});
  } else {
    if ((act & ~TF24_BIAS_F32) == TF24_ACT_RELU) output_pass(std::integral_constant<int, EPI_RELU>{});
    else if ((act & ~TF24_BIAS_F32) == TF24_ACT_SILU) output_pass(std::integral_constant<int, EPI_SILU>{});
    else output_pass(std::integral_constant<int, EPI_GELU>{});
  }
  if (!has_next) break;
  // ---- the next tile: its first two stages are (about to be) in the buffers nxt and fre
  i0 = next_i0; j0 = next_j0; chained = true;
  { const uint32_t t = cur; cur = nxt; nxt = fre; fre = t; }
#pragma unroll
  for (int ti = 0; ti < C::TI; ti++)
#pragma unroll
    for (int tj = 0; tj < C::TJ; tj++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[ti][tj][r] = 0;
  }
}

// Second pass of a split-K product: a block handles one eighth of a tile (the accumulator groups
// `slab` of one ti), same lane -> element mapping as spmm_pipe; sums the `splits` partial tiles
// (float32, or int32 for int8 operands) and applies scale / bias / activation / conversion.  SUMS: blocks past the tiles finish the
// row sums that a weight gradient's conversion left (a launch of their own takes 4 to 5 us; in a kernel of its own because the LDS that it
// takes costs the others 0.3 us).
template <typename Acc4, typename OutT, bool C_JMAJOR, typename C, bool SUMS>
__global__ void __launch_bounds__(C::THREADS)
spmm_reduce_splits(const float* __restrict__ partial, int splits, int tiles_i, int tiles_j, int64_t n_sparse, int64_t n_dense,
                   OutT* __restrict__ c, int64_t ldc, const OutT* __restrict__ bias, float scale, int act, RowSums sums) {
  const int ntiles = tiles_i * tiles_j;
  const int tile = blockIdx.x;
  if constexpr (SUMS) {
    if (tile >= ntiles) {
      row_sums_of_block(sums, (int64_t)(tile - ntiles) * gridDim.y + blockIdx.y);       // (past the last row: none)
      return;
    }
  }
  constexpr int GH = C::GH;
  const int group = tile / (GH * tiles_j);
  const int gh = min(GH, tiles_i - group * GH);
  const int in_group = tile - group * GH * tiles_j;
  const int64_t i0 = (int64_t)(group * GH + in_group % gh) * C::BI, j0 = (int64_t)(in_group / gh) * C::BJ;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wi = wave / C::WAVES_J, wj = wave % C::WAVES_J;
  const int l32 = lane & 31, lh = lane >> 5;
  constexpr int NSLAB = C::TI * C::TJ * 4;
  // gridDim.y blocks share the NSLAB accumulator groups of the tile
  for (int slab = blockIdx.y; slab < NSLAB; slab += gridDim.y) {
    const int ti = slab / (C::TJ * 4), tj = (slab / 4) % C::TJ, g = slab % 4;
    if (j0 + wj * C::WJ + tj * 32 >= n_dense) continue;          // the whole 32-column slab lies past the dense operand
    // the pieces are loaded eight at a time (independent loads in flight) and added in piece order
    Acc4 sum = {0, 0, 0, 0};
    const float* first = partial + (int64_t)tile * (C::BI * C::BJ) + ((int64_t)slab * C::THREADS + tid) * 4;
    const int64_t piece = (int64_t)ntiles * (C::BI * C::BJ);
    for (int sp0 = 0; sp0 < splits; sp0 += 8) {
      Acc4 part[8];
#pragma unroll
      for (int u = 0; u < 8; u++)
        part[u] = *reinterpret_cast<const Acc4*>(first + (int64_t)min(sp0 + u, splits - 1) * piece);
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (sp0 + u < splits) sum += part[u];
    }
    const int64_t col = j0 + wj * C::WJ + tj * 32 + l32;
    const int64_t row = i0 + wi * C::WI + ti * 32 + g * 8 + lh * 4;
    if (col >= n_dense || row >= n_sparse) continue;
    OutT o[4];
#pragma unroll
    for (int r = 0; r < 4; r++) o[r] = to_out<OutT>(finish_value(sum[r], scale, bias, row + r, act));
    if constexpr (C_JMAJOR) {
      *reinterpret_cast<Pack<OutT, 4>*>(c + col * ldc + row) = *reinterpret_cast<Pack<OutT, 4>*>(o);
    } else {
#pragma unroll
      for (int r = 0; r < 4; r++) c[(row + r) * ldc + col] = o[r];
    }
  }
}

// How many k pieces a product is cut into, for shapes whose tiles cannot fill the 256 compute units: the number for which
//     CALL_US + max(stages of one piece x STAGE_US, MB of the compressed operand x OPERAND_US)
//             + (pieces > 1: SPLIT_US + pieces x PIECE_US + MB of partial sums, all pieces, x PARTIAL_US) + (pieces > 8: 0.5),
// and 2 % more with over 208 blocks,
// is least, among those whose blocks fit one round of the compute units and whose float32 partial tiles fit the caller's
// workspace.  (Two of the narrowest tiles fit on one compute unit, but a few blocks more than there are units make the
// whole product wait for the shared ones: fp8 11008 x 11008 against 48 columns 19.3 us in 5 pieces = 215 blocks, 26.4 in 6 = 258.)
// Only the 32-column slabs that the dense operand reaches are written and read back, so only they count: k-strided
// 6144 x 1536 against 16 columns 20.5 us in one piece, 12.4 in five.  Below some pieces the narrowest tiles are bound by the
// one pass over the compressed operand (OPERAND_US: 8.8 TB/s, it stays in the last cache over repeated products).
// From nine pieces on the reduction, which loads eight at a time, goes round twice: 768 x 3072 against 86 columns 10.0 us in
// eight pieces, 10.5 in nine and more; 480 x 2816 against 321 11.7 in five, 13.2 in nine.
// Rounds of more than 208 blocks scatter: 4096 x 11008 against 257 to 305 columns 29.4 to 34.6 us in five pieces = 240 blocks,
// 29.8 to 30.8 in four.
// A stage of the smallest tiles takes longer the more units are busy (FULL_US) and the more both operands are (MEMORY_US a MB).
// The constants are least-squares fits, per tile configuration, to 25 000 timings of 1 to 16 pieces over fp16 and fp8 weights from
// 256 x 768 to 20480 x 11008 (6 to 512 stages) and 16 to 3072 dense columns.  The pieces chosen this way are within 1 % of
// the best ones on average and within 4 to 6 % for 19 in 20 (a fixed 192 / tiles of them: 5, 18 and 9 % off for the three
// configurations below, and twice the time at worst; a fit to the range of 768 x 768 to 8192 x 8192 alone that counted whole tiles
// 7, 2 and 5 %, half again the time at worst).  us, with 192 / tiles pieces and now: 3072 x 768 against 1024 columns
// 22.2 -> 9.0 (2 pieces -> 1), 4096 x 4096 against 128 19.0 -> 16.1 (12 -> 5); dW of 1024 tokens, 3072 x 768, 26.2 -> 16.4 (4 -> 1).
// A k-contiguous product of at most kShortStages stages is not cut: the reduction's launch and workspace are 4 us of host time,
// which bounds such calls one after the other (linear of 96 rows with 256 x 1536: 14.6 us a call in one piece, 18.5 in
// eight; alone 33.0 and 30.3 us, on the GPU 12.9 and 8.6).
struct PieceCost { double call_us, stage_us, split_us, piece_us, partial_us, operand_us, full_us = 0.0, memory_us = 0.0; };
template <typename C>
constexpr PieceCost piece_cost(bool k_strided) {
  return std::is_same<C, SmallCfg>::value ? PieceCost{4.63, 0.212, 1.86, 0.0, 0.545, 0.0, 0.025, 0.0013}
         : std::is_same<C, SlimCfg>::value ? PieceCost{3.96, 0.172, 1.99, 0.0, 0.511, 0.136, 0.0, 0.0008}
         : std::is_same<C, TallSlimCfg>::value ? PieceCost{5.1, 0.37, 1.8, 0.0, 0.48, 0.113}
         : std::is_same<C, MidCfg>::value ? PieceCost{5.6, 0.33, 2.1, 0.1, 0.45, 0.0}
         : std::is_same<C, SquareCfg>::value ? PieceCost{7.3, 0.40, 1.15, 0.0, 0.40, 0.0}
         : k_strided ? PieceCost{7.1, 0.55, 1.15, 0.0, 0.42, 0.0} : PieceCost{6.9, 0.50, 3.3, 0.0, 0.385, 0.0};
}
constexpr int64_t kShortStages = 28;
struct Pieces { int count; double us; };
template <typename T, typename C>
Pieces choose_pieces(int64_t n_sparse, int64_t k, int64_t n_dense, int64_t workspace_bytes, bool k_strided) {
  const PieceCost cost = piece_cost<C>(k_strided);
  const int64_t tiles_i = (n_sparse + C::BI - 1) / C::BI, tiles = tiles_i * ((n_dense + C::BJ - 1) / C::BJ);
  const int64_t stages = k * (int64_t)sizeof(T) / C::KB;
  const double operand_us = (double)(n_sparse * k * (int64_t)sizeof(T)) * (9.0 / 16.0) * 1e-6 * cost.operand_us;
  const double partial_us = (double)(tiles_i * C::BI * ((n_dense + 31) / 32 * 32)) * 4e-6 * cost.partial_us;     // of one piece
  const double memory_us = ((double)(n_sparse * k) * (9.0 / 16.0) + (double)(n_dense * k)) * (double)sizeof(T) * 1e-6 * cost.memory_us;
  auto us = [&](int64_t p) {
    const double stage_us = cost.stage_us + (double)(p * tiles) / 256.0 * cost.full_us + memory_us;
    const double one = cost.call_us + std::max((double)((stages + p - 1) / p) * stage_us, operand_us);
    if (p == 1) return one;
    return (one + cost.split_us + (double)p * (cost.piece_us + partial_us) + (p > 8 ? 0.5 : 0.0)) * (p * tiles > 208 ? 1.02 : 1.0);
  };
  Pieces best{1, us(1)};
  if (!k_strided && stages <= kShortStages) return best;
  for (int64_t p = 2; p <= 16 && p <= stages / 2 && p * tiles <= 256 && p * tiles * C::BI * C::BJ * 4 <= workspace_bytes; p++)
    if (us(p) < best.us) best = {(int)p, us(p)};
  return best;
}

// At most 64 columns: whether 256 x 64 tiles instead of 128 x 64 ones, of which a compute unit holds two of either.  By the rows of 128 x 64 tiles there are
// (620 products of 129 to 2112 of them and 2 to 256 stages, fp16 and e4m3; us on 128 x 64 and on 256 x 64 tiles, operands from memory):
// 129 to 168: the former are one piece of k (two are slower throughout: 1.02 to 1.7 times), of the latter there is room for three.  That pays where k is long, the
// longer the more of the units one piece fills: fp16 16416 x 8192 against 64 columns 43.3 and 38.5, 18880 x 14336 77.9 and 63.0, but 16416 x 4096 23.7 and 25.9,
// 20480 x 8192 43.5 and 46.0.  (With the weight in the caches it pays some 80 stages later: e4m3 18912 x 18944 35.4 and 41.9, from memory 51.4 and 47.7.)
// 169 to 256: 128 x 64 throughout, 1.1 to 1.5 times as fast (28544 x 4032 25.7 and 40.1).
// 257 to 512: units with two tiles of the one kind beside units with one, or one of the other kind each: fp16 32832 x 5056 58.2 and 53.7, e4m3 34560 x 11136
// 67.2 and 56.5, 62592 x 768 15.6 and 13.9, but under 12 stages no better (47584 x 192 5.9 and 6.5; 36128 x 576 10.2 and 9.7, from the caches 6.3 and 7.9).
// Beyond that the rounds are full with either, and the smaller tiles are the faster ones (e4m3 by a fifth) unless the others' last round is
// three quarters full or more and the values are of 16 bits: fp16 114976 x 320 13.4 and 11.4, 128256 x 2048 63.9 and 59.0, 247104 x 320 28.7 and 25.3.
constexpr int64_t kTallSlimMinStages = 12;
inline bool takes_tall_slim(int64_t n_sparse, int64_t stages, bool eight_bit) {
  const int64_t rows = (n_sparse + SlimCfg::BI - 1) / SlimCfg::BI;
  if (rows <= 128) return false;
  if (rows <= 256) return rows <= 168 && stages >= 100 + (rows - 128) * 5 / 2;
  if (rows <= 512) return stages >= kTallSlimMinStages;
  return !eight_bit && (rows - 1) % 1024 >= 768;
}

// A k-contiguous dense operand of more than 64 columns takes 256 x 128 tiles up to 128 columns, and beyond that where they fit one
// round of the 256 compute units: they reach twice as many of them as 256 x 256 tiles, which are then the faster ones only with
// k pieces under a long k (of 671 products timed with the pieces chosen above: 4096 x 4096 against 1000 columns
// 30.0 and 43.2 us, 1600 x 6400 against 3000 48.1 and 59.9, but 6144 x 32768 against 512 159 and 118; with this
// comparison of the estimates no product is more than 2 % off the better of the two, without it 4 are, by up to 35 %).
template <typename T>
bool takes_mid(int64_t n_sparse, int64_t k, int64_t n_dense, int64_t workspace_bytes) {
  if (n_dense <= MidCfg::BJ) return true;
  if (((n_sparse + MidCfg::BI - 1) / MidCfg::BI) * ((n_dense + MidCfg::BJ - 1) / MidCfg::BJ) > 256) return false;
  return n_dense < TiledCfg::BJ || choose_pieces<T, TiledCfg>(n_sparse, k, n_dense, workspace_bytes, false).us >=
                                       0.95 * choose_pieces<T, MidCfg>(n_sparse, k, n_dense, workspace_bytes, false).us;
}

// More than 64 columns (k-contiguous) take 128 x 128 tiles where one round of the compute units holds them and the estimate for them is below that of
// the tiles above.  Of 220 products of 256 to 12288 rows, 2 to 320 stages and 72 to 4008 columns (fp16 and e4m3) 200 take them, 15 % less time
// on average over all; the choice is 0.5 % off the better one on average.  us, then and now: fp16 768 x 768 against
// 160 columns 8.6 and 6.8, 3072 x 768 against 952 9.2 and 7.6, 1600 x 1600 against 1792 13.4 and 10.8, 4096 x 4096 against 128 16.0 and
// 14.4, against 512 23.1 and 20.7, 6144 x 4096 against 424 28.9 and 21.5; e4m3 8192 x 8192 against 480 41.6 and 28.2.  The other way round, where
// the operands no longer fit the caches: 5824 x 10176 against 328 47 and 63, 2048 x 20480 against 760 57 and 81.  More than one round:
// 5120 x 1280 against 840 (280 tiles) 13.1 and 16.3 with two tiles to a unit.
// The estimates are of operands in the caches.  From memory a stage of these tiles takes 0.4 us, whatever their number (three stages are under way, for
// 1.2 us), so one piece of a long k is the slower way where the others' is cut: of 450 such products those above kColdPart times the others' estimate lose 8 %
// on average over both operands from memory, the weight alone and neither; us there on the other tiles and on these fp16 1600 x 6400 against 1296 columns 33.9, 34.7,
// 30.3 and 44.1, 38.9, 30.4, e4m3 4096 x 11008 against 457 30.7, 29.5, 25.2 and 40.5, 32.4, 27.5.  Those below it gain 4, 13 and 15 %, a sixth of them for a loss from
// memory: 1024 x 4096 against 1455 25.2, 20.6, 20.5 and 30.5, 19.6, 19.6.
constexpr double kColdStageUs = 0.4, kColdPart = 1.35;
template <typename T>
bool takes_small(int64_t n_sparse, int64_t k, int64_t n_dense, int64_t workspace_bytes) {
  if (n_dense <= SlimCfg::BJ || ((n_sparse + SmallCfg::BI - 1) / SmallCfg::BI) * ((n_dense + SmallCfg::BJ - 1) / SmallCfg::BJ) > 256) return false;
  const Pieces others = takes_mid<T>(n_sparse, k, n_dense, workspace_bytes) ? choose_pieces<T, MidCfg>(n_sparse, k, n_dense, workspace_bytes, false)
                                                                           : choose_pieces<T, TiledCfg>(n_sparse, k, n_dense, workspace_bytes, false);
  const Pieces small = choose_pieces<T, SmallCfg>(n_sparse, k, n_dense, workspace_bytes, false);
  const double cold_us = piece_cost<SmallCfg>(false).call_us + kColdStageUs * (double)(k * (int64_t)sizeof(T) / SmallCfg::KB);
  return small.us < others.us && !(small.count == 1 && others.count > 1 && cold_us > kColdPart * others.us);
}

// Between the two: a product whose 128 x 128 tiles are more than one round of the compute units and whose 192 x 128 ones are not takes the latter instead of
// 256 x 128 ones.  It is in one piece (more than half a round of any of these tiles), so again its time is that of a tile, with 3/4 of the stages' work.
// From 20 stages on (below, the longer ring and the third of the rounds that the wider tiles leave empty weigh as much: 60 products, us on 256 x 128
// and on these tiles 2304 x 768 against 2368 columns 10.6 and 11.3, 768 x 768 against 6048 9.6 and 9.3) up to 176 (operands that no longer
// fit the caches: 172 stages 4096 x 11008 against 936 70.2 and 66.0, 189 5952 x 12096 against 784 95 and 100).  Between them 37 of 39 products are
// faster and two within 2 %, 9 % less time on average: 3840 x 1280 against 1040 13.6 and 12.4, 6144 x 4096 against 736 34.1 and 30.1, 11008 x 4096 against
// 336 40.7 and 32.6, 2048 x 8192 against 2928 79.7 and 65.7; e4m3 12288 x 4096 against 320 17.7 and 16.3.
constexpr int64_t kLowerMinStages = 20, kLowerMaxStages = 176;
template <typename T>
bool takes_lower(int64_t n_sparse, int64_t k, int64_t n_dense, int64_t workspace_bytes) {
  const int64_t columns = (n_dense + LowerCfg::BJ - 1) / LowerCfg::BJ;
  const int64_t stages = k * (int64_t)sizeof(T) / LowerCfg::KB;
  return stages >= kLowerMinStages && stages <= kLowerMaxStages && n_dense > LowerCfg::BJ && ((n_sparse + SmallCfg::BI - 1) / SmallCfg::BI) * columns > 256 &&
         ((n_sparse + LowerCfg::BI - 1) / LowerCfg::BI) * columns <= 256 && takes_mid<T>(n_sparse, k, n_dense, workspace_bytes);
}

// Rounds of the compute units that so many tiles take (each XCD has an eighth of both).
inline int64_t tile_rounds(int64_t tiles, int64_t cu_slots) { return ((tiles + 7) / 8 + cu_slots - 1) / cu_slots; }

// A last round that fills less than half of the compute units: the tile rows that make up the full rounds stay
// with the chained 256 x 256 tiles, the remaining rows go to a second launch on 256 x 128 tiles, which reach twice
// as many compute units for half the time each (fp16, W[11008, 4096] against 8192 tokens, before 384 x 192 tiles took that
// product (takes_tall): 1376 tiles = 5 rounds of 256 + 96; 40 tile rows chained, 3 rows as 192 half tiles: 351.6 -> 341.6 us;
// e4m3, W[8448, 8192] against 8192: 291 -> 277).  Long tiles only: what a short tile's round costs is mostly its prologue and
// output pass, which the second launch pays again.
struct TileRows { int tiles_i, tail_rows; };
inline TileRows full_rounds(int64_t n_sparse, int64_t n_dense, int stages, int cu_slots) {
  const int tiles_i = (int)((n_sparse + TiledCfg::BI - 1) / TiledCfg::BI), tiles_j = (int)((n_dense + TiledCfg::BJ - 1) / TiledCfg::BJ);
  const int cus = cu_slots * 8, tiles = tiles_i * tiles_j;
  if (cus <= 0 || tiles % cus == 0 || stages < kWave4MinStages) return {tiles_i, 0};
  const int rows = tiles / cus * cus / tiles_j, left = tiles_i - rows;                       // tile rows of the full rounds
  const int64_t half_tiles = (int64_t)left * ((n_dense + MidCfg::BJ - 1) / MidCfg::BJ);
  return rows * tiles_j > cus && left > 0 && half_tiles <= cus ? TileRows{rows, left} : TileRows{tiles_i, 0};
}

// Whether a product with 16-bit j-major results and k contiguous, in one piece, takes 192 x 192 tiles: rounds x (us of a tile's
// stages + its prologue and output pass) against the same of what it would take otherwise -- 256 x 256 tiles (chained, with
// their last rows on half tiles: full_rounds), or from kWave4MinStages stages on 256 x 192 ones.  Where full rounds follow each
// other the matrix cores are held to the clock that their power allows, and no tile takes less than its share of the chip at that
// clock: 0.67 us a stage of 256 square tiles, 0.75 and 1.0 of the others, whose fragments serve more instructions.  Of 258
// products of 5 to 172 stages drawn from 512 to 11008 rows and 500 to 16000 columns (fp16, bf16 and e4m3, operands that change
// from product to product) the choice is 0.04 % off the better one on average, 3.6 % at worst; of 90 others that the constants
// were not fitted to, a third of them on the same operands, 0.01 and 0.6 %.  (With 0.53 and 1.6 for square tiles and 0.88 and 3.8
// for the 8-wave ones, which were read off few products, 2.2 and 18 % below 32 stages: 3072 x 768 against 12288 columns 44.2 us
// on wide tiles and 48.3 on square ones, 2048 x 512 23.9 and 27.9, 6656 x 704 against 12879 86 and 101.)
inline bool takes_square(int64_t n_sparse, int64_t n_dense, int stages, TileRows wide, int cu_slots) {
  const int64_t tiles_j = (n_dense + TiledCfg::BJ - 1) / TiledCfg::BJ;
  const int64_t square = ((n_sparse + SquareCfg::BI - 1) / SquareCfg::BI) * ((n_dense + SquareCfg::BJ - 1) / SquareCfg::BJ);
  const bool four_waves = stages >= kWave4MinStages;
  auto us = [&](int64_t tiles, double of_round, double sustained) {
    return std::max((double)tile_rounds(tiles, cu_slots) * of_round, (double)tiles / (8 * cu_slots) * sustained * stages);
  };
  double others = us(wide.tiles_i * tiles_j, four_waves ? 0.93 * stages + 2.5 : 0.84 * stages + 5.5, 1.0);
  if (wide.tail_rows) others += 0.5 * stages + 5.0;
  if (four_waves) {
    const int64_t narrow = (wide.tiles_i + wide.tail_rows) * ((n_dense + Wave4Cfg192::BJ - 1) / Wave4Cfg192::BJ);
    others = std::min(others, us(narrow, 0.69 * stages + 2.0, 0.75));
  }
  return us(square, 0.53 * stages + 5.0, 0.67) < 0.95 * others;
}

// The tiles of a product with j-major results and k contiguous, in one piece: 256 x 256 ones on eight waves, or 4-wave forms --
// those, where there are more of them than compute units (chained), 256 x 192 or 192 x 192 ones (16-bit results).
// 256 x 192 also where both widths fit one round and the narrow tiles spread over more compute units (W[768, 3072] against
// 12288 tokens: 144 wide tiles or 192 narrow ones, 36.1 -> 34.1 us; W[1024, 4096]: 192 or 256 tiles, 56.2 -> 53.9 us).
enum class Tiles { WIDE8, WIDE4, NARROW4, SQUARE4, TALL4 };
inline Tiles choose_without_tall(int64_t n_sparse, int64_t n_dense, int stages, TileRows wide, bool results16, int cu_slots) {
  if (results16 && takes_square(n_sparse, n_dense, stages, wide, cu_slots)) return Tiles::SQUARE4;
  if (stages < kWave4MinStages) return Tiles::WIDE8;
  const int64_t tiles = wide.tiles_i * ((n_dense + TiledCfg::BJ - 1) / TiledCfg::BJ), narrow = wide.tiles_i * ((n_dense + Wave4Cfg192::BJ - 1) / Wave4Cfg192::BJ);
  const int64_t rounds = tile_rounds(tiles, cu_slots), narrow_rounds = tile_rounds(narrow, cu_slots);
  if (results16 && narrow_rounds <= rounds && (narrow_rounds > 1 || (narrow + 7) / 8 > (tiles + 7) / 8)) return Tiles::NARROW4;
  return rounds > 1 ? Tiles::WIDE4 : Tiles::WIDE8;
}

// Whether it takes 384 x 192 tiles instead of the form chosen among the others: the same estimate of both (0.98 us a stage and 5 us
// for a round of these tiles, 1.12 a stage at the sustained clock), from kWave4MinStages stages on (choose_short: fewer).  Of 110 fp16 products of 10 to 168
// stages, 960 to 12224 rows and 1237 to 15757 columns on operands that change from product to product, 13 take them, all 2 to 28 %
// faster that way (1120 x 2816 against 14480 columns 69.9 -> 54.8, 2912 x 5824 against 12074 244 -> 200, 10624 x 3264 against 3385
// 132 -> 117); of the others none would be more than 5 % faster.  Of 70 others, a third with bias, half of them bf16, 12
// take them, 1 to 25 % faster.
inline bool takes_tall(int64_t n_sparse, int64_t n_dense, int stages, TileRows wide, Tiles form, int cu_slots) {
  auto us = [&](int64_t tiles, double of_round, double sustained) {
    return std::max((double)tile_rounds(tiles, cu_slots) * of_round, (double)tiles / (8 * cu_slots) * sustained * stages);
  };
  auto columns = [&](int64_t width) { return (n_dense + width - 1) / width; };
  auto rows = [&](int64_t height) { return (n_sparse + height - 1) / height; };
  double other;
  if (form == Tiles::SQUARE4) other = us(rows(SquareCfg::BI) * columns(SquareCfg::BJ), 0.53 * stages + 5.0, 0.67);
  else if (form == Tiles::NARROW4) other = us(rows(Wave4Cfg192::BI) * columns(Wave4Cfg192::BJ), 0.69 * stages + 2.0, 0.75);
  else other = us(wide.tiles_i * columns(TiledCfg::BJ), 0.93 * stages + 2.5, 1.0) +
               (wide.tail_rows ? 0.5 * stages + 5.0 : 0.0);
  return us(rows(TallCfg::BI) * columns(TallCfg::BJ), 0.98 * stages + 5.0, 1.12) < 0.98 * other;
}

// Whether a product of fewer than kWave4MinStages stages takes 256 x 192 or (16-bit operands, kShortTallMinStages stages or more) 384 x 192 tiles
// instead of the form chosen among the others.  Rounds and filled rounds (tiles / compute units) each cost something by the stage and by the tile;
// fitted to the times of every form on 230 products of 5 to 31 stages (fp16, bf16 and e4m3, 640 to 11000 rows, 900 to 16000 columns,
// operands that change from product to product), within 5 % of them (root mean square).  97 of those products take the two forms, 6 % faster on
// average, 17 % at best and 9 % slower at worst; over all of them the choice is 0.6 % off the best form.  us on the others and now: fp16
// 3072 x 768 against 12288 columns (three full rounds of 256 x 192 tiles) 41.8 and 39.0, 5120 x 1280 against 4096 40.0 and 36.2, 4800 x 1600
// against 4096 47.0 and 41.9, 4096 x 960 against 4145 26.1 and 23.3 (384 x 192).  One round of wide tiles and of narrow ones, up to 11 stages:
// no better (2048 x 512 against 6144 13.1 and 13.6, e4m3 4224 x 1024 against 2384 12.1 and 14.6; with 12 stages 2304 x 768 against 4096 14.3 and 13.7).
constexpr int kShortTallMinStages = 8, kShortOneRoundStages = 12;
inline Tiles choose_short(int64_t n_sparse, int64_t n_dense, int stages, Tiles form, bool operands16, int cu_slots) {
  struct Cost { int rows, columns; double round_stage, stage, round, tile, call; };
  auto rounds_of = [&](int rows, int columns) { return tile_rounds(((n_sparse + rows - 1) / rows) * ((n_dense + columns - 1) / columns), cu_slots); };
  auto us = [&](Cost c) {
    const double filled = (double)(((n_sparse + c.rows - 1) / c.rows) * ((n_dense + c.columns - 1) / c.columns)) / (8 * cu_slots);
    return (double)rounds_of(c.rows, c.columns) * (c.round_stage * stages + c.round) + filled * (c.stage * stages + c.tile) + c.call;
  };
  const Cost wide{TiledCfg::BI, TiledCfg::BJ, 0.37, 0.56, 2.49, 1.85, 2.81}, square{SquareCfg::BI, SquareCfg::BJ, 0.34, 0.23, 2.9, 0.0, 3.52};
  const Cost present = form == Tiles::SQUARE4 ? square : wide;
  const double other = us(present), narrow = us({Wave4Cfg192::BI, Wave4Cfg192::BJ, 0.33, 0.37, 4.3, 0.0, 2.31});
  const double tall = us({TallCfg::BI, TallCfg::BJ, 0.52, 0.40, 4.48, 4.37, 1.3});
  if (operands16 && stages >= kShortTallMinStages && tall < 0.96 * narrow) return tall < 0.98 * other ? Tiles::TALL4 : form;
  if (stages < kShortOneRoundStages && rounds_of(present.rows, present.columns) == 1) return form;
  return narrow < 0.98 * other ? Tiles::NARROW4 : form;
}
inline Tiles choose_tiles(int64_t n_sparse, int64_t n_dense, int stages, TileRows wide, bool results16, int cu_slots, bool operands16 = false) {
  if (cu_slots <= 0 || stages < 4) return Tiles::WIDE8;
  const Tiles form = choose_without_tall(n_sparse, n_dense, stages, wide, results16, cu_slots);
  if (results16 && stages < kWave4MinStages) return choose_short(n_sparse, n_dense, stages, form, operands16, cu_slots);
  return results16 && operands16 && takes_tall(n_sparse, n_dense, stages, wide, form, cu_slots) ? Tiles::TALL4 : form;
}

// Whether a product with k strided does: the pieces that either tile would be cut into, estimated as choose_pieces does and
// with further rounds counted by their stages.  (Few products are not: 6400 x 2816 against 1600 columns, 306 tiles instead of 175,
// 39.8 us and 45.  Uncut 16-bit results stored i-major would leave in 2-byte stores: the staged pass takes 64 columns.)
template <typename T, typename OutT>
bool strided_takes_square(int64_t n_sparse, int64_t k, int64_t n_dense, int64_t workspace_bytes, bool c_jmajor, int cu_slots) {
  if (cu_slots <= 0) return false;
  const int64_t stages = k * (int64_t)sizeof(T) / TiledCfg::KB;
  auto us = [&](auto cfg, Pieces p) {
    using C = decltype(cfg);
    const int64_t tiles = ((n_sparse + C::BI - 1) / C::BI) * ((n_dense + C::BJ - 1) / C::BJ);
    return p.us + (double)((tile_rounds(tiles * p.count, cu_slots) - 1) * ((stages + p.count - 1) / p.count)) * piece_cost<C>(true).stage_us;
  };
  const Pieces wide = choose_pieces<T, TiledCfg>(n_sparse, k, n_dense, workspace_bytes, true);
  const Pieces square = choose_pieces<T, SquareCfg>(n_sparse, k, n_dense, workspace_bytes, true);
  if (sizeof(OutT) == 2 && !c_jmajor && square.count == 1) return false;
  return us(SquareCfg{}, square) < 0.97 * us(TiledCfg{}, wide);
}

template <typename T, typename OutT, typename C>
int launch_tiled(const void* av, const void* am, int64_t n_sparse, int64_t k, const void* b, int b_layout, int64_t ldb,
                 int64_t n_dense, void* c, int c_layout, int64_t ldc, const void* bias, float scale, int act,
                 void* workspace, int64_t workspace_bytes, hipStream_t s, RowSums* sums = nullptr) {
  constexpr bool SQUARE = std::is_same<C, SquareCfg>::value;       // (this way for a k-strided dense operand only)
  const int cu_slots = compute_units() / 8;
  if constexpr (std::is_same<C, TiledCfg>::value && sizeof(T) == 2) {
    if (b_layout == TF24_COL_MAJOR &&
        strided_takes_square<T, OutT>(n_sparse, k, n_dense, workspace ? workspace_bytes : 0, c_layout == TF24_COL_MAJOR, cu_slots))
      return launch_tiled<T, OutT, SquareCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace,
                                              workspace_bytes, s, sums);
  }
  int tiles_i = (int)((n_sparse + C::BI - 1) / C::BI);
  const int tiles_j = (int)((n_dense + C::BJ - 1) / C::BJ);
  const int splits = workspace && !std::is_same<C, LowerCfg>::value ? choose_pieces<T, C>(n_sparse, k, n_dense, workspace_bytes, b_layout == TF24_COL_MAJOR).count : 1;
  const int stages = (int)(k * (int64_t)sizeof(T) / C::KB);
  int tail_rows = 0;
  if constexpr (std::is_same<C, TiledCfg>::value) {
    if (c_layout == TF24_COL_MAJOR && b_layout == TF24_ROW_MAJOR && splits == 1) {
      const TileRows rows = full_rounds(n_sparse, n_dense, stages, cu_slots);
      tiles_i = rows.tiles_i;
      tail_rows = rows.tail_rows;
    }
  }
  const int per_xcd = (tiles_i * tiles_j * splits + 7) / 8;
  // More tiles than compute units and no k pieces: one workgroup per compute unit walks its tiles in
  // one pipeline (the next tile's operands arrive while the current one is written out).
  const bool persist = C::BJ == 256 && c_layout == TF24_COL_MAJOR && splits == 1 &&
                       k * (int64_t)sizeof(T) / C::KB >= 4 && per_xcd > cu_slots && cu_slots > 0;
  dim3 grid((unsigned)((persist ? cu_slots : per_xcd) * 8));
  const bool jm = c_layout == TF24_COL_MAJOR;
  // Start stagger of chained tiles (see spmm_pipe): half an output burst -- 256 tiles of 128 KB (16-bit) or 256 KB
  // (32-bit) at the HBM write rate are 6 or 12 us -- for short tiles, whose time the bursts are a large part of, and
  // for 32-bit outputs over three or more rounds.  Measured: 576 tiles of 12 stages 48.9 -> 43.4 us (the training
  // step they belong to 0.684 -> 0.679 ms), 2048 tiles of 64 fp8 stages with float32 output 0.521 -> 0.514 ms; with
  // 16-bit outputs the same tiles are unchanged and 1376 tiles of 64 fp16 stages lose 0.2 % (alternating with another
  // product; 1.6 % faster when the same product repeats), so long 16-bit tiles start together.
  const int stagger_rounds = persist ? (per_xcd + cu_slots - 1) / cu_slots : 0;
  const int stagger = !persist ? 0 : k * (int64_t)sizeof(T) / C::KB <= 32 ? (sizeof(OutT) == 2 ? 300 : 600)
                               : (sizeof(OutT) == 4 && stagger_rounds >= 3) ? 600 : 0;
  const Tiles form = std::is_same<C, TiledCfg>::value && jm && b_layout == TF24_ROW_MAJOR && splits == 1
                         ? choose_tiles(n_sparse, n_dense, stages, {tiles_i, tail_rows}, sizeof(OutT) == 2, cu_slots, sizeof(T) == 2) : Tiles::WIDE8;
  auto launch_tail = [&]() {                       // the rows behind the full rounds, on 256 x 128 tiles
    if constexpr (std::is_same<C, TiledCfg>::value) {
      if (tail_rows > 0) {
        const int tj = (int)((n_dense + MidCfg::BJ - 1) / MidCfg::BJ);
        const dim3 tgrid((unsigned)((tail_rows * tj + 7) / 8 * 8));
        auto tail = [&](auto acts) {
          hipLaunchKernelGGL((spmm_pipe<T, OutT, true, MidCfg, false, false, decltype(acts)::value>), tgrid, dim3(MidCfg::THREADS), 0, s,
                             (const uint8_t*)av, (const uint8_t*)am, n_sparse, k, (const uint8_t*)b, ldb * (int64_t)sizeof(T), n_dense,
                             (OutT*)c, ldc, (const OutT*)bias, scale, act, tail_rows, tj, 1, (float*)nullptr, tiles_i);
        };
        if ((act & ~TF24_BIAS_F32) == TF24_ACT_NONE) tail(std::false_type{}); else tail(std::true_type{});
      }
    }
  };
  if constexpr (std::is_same<C, TiledCfg>::value && sizeof(OutT) == 2) {
    auto chained = [&](auto cfg, auto acts, int ti, int tj, int start_stagger) {
      using Cfg = decltype(cfg);
      hipLaunchKernelGGL((spmm_pipe<T, OutT, true, Cfg, false, true, decltype(acts)::value>), dim3((unsigned)(cu_slots * 8)), dim3(Cfg::THREADS), 0, s,
                         (const uint8_t*)av, (const uint8_t*)am, n_sparse, k, (const uint8_t*)b, ldb * (int64_t)sizeof(T), n_dense,
                         (OutT*)c, ldc, (const OutT*)bias, scale, act, ti, tj, 1, (float*)nullptr, start_stagger);
    };
    auto either = [&](auto cfg, int ti, int tj, int start_stagger) {
      if ((act & ~TF24_BIAS_F32) == TF24_ACT_NONE) chained(cfg, std::false_type{}, ti, tj, start_stagger);
      else chained(cfg, std::true_type{}, ti, tj, start_stagger);
    };
    if (form == Tiles::SQUARE4) {
      const int ti = (int)((n_sparse + SquareCfg::BI - 1) / SquareCfg::BI), tj = (int)((n_dense + SquareCfg::BJ - 1) / SquareCfg::BJ);
      either(SquareCfg{}, ti, tj, tile_rounds((int64_t)ti * tj, cu_slots) > 1 && stages <= 32 ? 300 : 0);
      return check_launch("tf24_spmm");
    }
    if constexpr (sizeof(T) == 2) {
      if (form == Tiles::TALL4) {
        either(TallCfg{}, (int)((n_sparse + TallCfg::BI - 1) / TallCfg::BI), (int)((n_dense + TallCfg::BJ - 1) / TallCfg::BJ), 0);
        return check_launch("tf24_spmm");
      }
    }
    if (form == Tiles::NARROW4) {
      either(Wave4Cfg192{}, tiles_i, (int)((n_dense + Wave4Cfg192::BJ - 1) / Wave4Cfg192::BJ), stagger);
      launch_tail();
      return check_launch("tf24_spmm");
    }
  }
  auto launch_epi = [&](auto c_jmajor, auto b_kstrided, auto acts) {
    constexpr bool ACTS = decltype(acts)::value;
    if constexpr (C::BJ == 256 && decltype(c_jmajor)::value) {
      if constexpr (std::is_same<C, TiledCfg>::value && !decltype(b_kstrided)::value) {
        if (form == Tiles::WIDE4) {
          hipLaunchKernelGGL((spmm_pipe<T, OutT, true, Wave4Cfg, false, true, ACTS>), grid, dim3(Wave4Cfg::THREADS), 0, s,
                             (const uint8_t*)av, (const uint8_t*)am, n_sparse, k, (const uint8_t*)b, ldb * (int64_t)sizeof(T), n_dense,
                             (OutT*)c, ldc, (const OutT*)bias, scale, act, tiles_i, tiles_j, splits, (float*)workspace, stagger);
          return;
        }
      }
      if (persist) {
        hipLaunchKernelGGL((spmm_pipe<T, OutT, decltype(c_jmajor)::value, C, decltype(b_kstrided)::value, true, ACTS>), grid, dim3(C::THREADS), 0, s,
                           (const uint8_t*)av, (const uint8_t*)am, n_sparse, k, (const uint8_t*)b, ldb * (int64_t)sizeof(T), n_dense,
                           (OutT*)c, ldc, (const OutT*)bias, scale, act, tiles_i, tiles_j, splits, (float*)workspace, stagger);
        return;
      }
    }
    hipLaunchKernelGGL((spmm_pipe<T, OutT, decltype(c_jmajor)::value, C, decltype(b_kstrided)::value, false, ACTS>), grid, dim3(C::THREADS), 0, s,
                       (const uint8_t*)av, (const uint8_t*)am, n_sparse, k, (const uint8_t*)b, ldb * (int64_t)sizeof(T), n_dense,
                       (OutT*)c, ldc, (const OutT*)bias, scale, act, tiles_i, tiles_j, splits, (float*)workspace, 0);
  };
  auto launch = [&](auto c_jmajor, auto b_kstrided) {
    // with k pieces the reduction kernel applies bias and activation, not this one
    if ((act & ~TF24_BIAS_F32) == TF24_ACT_NONE || splits > 1) launch_epi(c_jmajor, b_kstrided, std::false_type{});
    else launch_epi(c_jmajor, b_kstrided, std::true_type{});
  };
  bool kstrided = SQUARE;
  if constexpr (sizeof(T) == 2 && C::BJ == 256) kstrided = b_layout == TF24_COL_MAJOR;
  if (kstrided) {
    if constexpr (sizeof(T) == 2 && (C::BJ == 256 || SQUARE)) {
      if (jm) launch(std::true_type{}, std::true_type{});
      else launch(std::false_type{}, std::true_type{});
    }
  } else if constexpr (!SQUARE) {
    if (jm) launch(std::true_type{}, std::false_type{});
    else launch(std::false_type{}, std::false_type{});
  }
  launch_tail();
  if (splits > 1) {
    constexpr int GROUPS = C::TI * C::TJ * 4;                                      // one accumulator group of the tile per block
    auto reduce = [&](auto c_jmajor, auto with_sums, const RowSums& rows) {
      hipLaunchKernelGGL((spmm_reduce_splits<typename mma32<T>::acc4_t, OutT, decltype(c_jmajor)::value, C, decltype(with_sums)::value>),
                         dim3((unsigned)(tiles_i * tiles_j + (rows.blocks() + GROUPS - 1) / GROUPS), GROUPS), dim3(C::THREADS), 0, s, (const float*)workspace, splits,
                         tiles_i, tiles_j, n_sparse, n_dense, (OutT*)c, ldc, (const OutT*)bias, scale, act, rows);
    };
    // The row sums go with the tiles that a weight gradient takes; from any other product they come back as they are, and the caller finishes them.
    bool added = false;
    if constexpr (sizeof(T) == 2 && (std::is_same<C, TiledCfg>::value || SQUARE)) {
      if (sums && !jm) {
        reduce(std::false_type{}, std::true_type{}, *sums);
        sums->partial = nullptr;                                                  // (finished here)
        added = true;
      }
    }
    if (!added) {
      if (jm) reduce(std::true_type{}, std::false_type{}, RowSums{});
      else reduce(std::false_type{}, std::false_type{}, RowSums{});
    }
  }
  return check_launch("tf24_spmm");
}

// ------------------------------------------------------------------------------------------
// Narrow kernels: at most 64 dense columns (decoding a few tokens against a large sparse weight, a batch of
// sequences against a small one).
// The product is bound by one pass over the compressed operand, so the sparse operand is not
// staged: a wave streams the A fragments of 16 sparse rows straight into registers (in the panel
// layout 1 KB of contiguous memory per panel, 16 bytes per lane, and their index words 128 (256)
// contiguous bytes) and runs one V_SMFMAC_*_16X16 per panel.  Loads are issued a batch of panels at
// a time into one of two register sets, the next batch while the current one is multiplied: left
// to itself the compiler waits for each panel's loads before it issues the next.
// A batch that reaches past the last panel re-reads it and leaves it out of the product: multiplied by zeros it would
// make NaN of an infinite activation.  The full batches are straight-line code and only the last one tests its panels,
// which is also the faster form (with a test of zeros in every panel 1600 x 6400 fp16 against one column takes 8.5 us, with
// a choice of the two forms in every batch 9.3, this way 7.8).
// Up to 32 columns mostly (takes_few): spmm_few.  Others (spmm_narrow): a block owns 16 rows, its up to four waves each take a
// share of the k range, read their dense fragments, NB of 16 columns, from global memory (64 contiguous bytes from
// each of the 16 dense rows, twice) and meet in LDS at the end (added in wave order).  Bound by latency, a few loads deep, at
// short k and by the requests of the dense fragments at long k: 3072 x 768 bf16 against 37 columns 5.7 us on 128 x 64 tiles,
// of which there are 24, and 5.0 us here.
// ------------------------------------------------------------------------------------------
constexpr int kNarrowWaves = 4;
// us on spmm_narrow and on spmm_few, 24 columns fp16: 2048 x 512 (8 panels) 3.7 and 3.8, 640 x 640 3.8 and 4.1, 3072 x 768 4.4 and 4.1, 1600 x 1600 6.0 and 4.8
constexpr int64_t kFewPanels = 12;
template <typename T, typename OutT, bool C_JMAJOR, int NB>
__global__ void __launch_bounds__(64 * kNarrowWaves)
spmm_narrow(const uint8_t* __restrict__ a_values, const uint8_t* __restrict__ a_meta, int64_t n_sparse, int64_t k,
            const uint8_t* __restrict__ b, int64_t ldb_bytes, int64_t n_dense,
            OutT* __restrict__ c, int64_t ldc, const OutT* __restrict__ bias, float scale, int act) {
  constexpr int KSTEP = mma16<T>::KSTEP;     // dense k per panel = per instruction
  constexpr int M_ROW = KSTEP / 8;           // metadata bytes per row per panel
  constexpr int BATCH = NB == 1 ? 8 : NB == 2 ? 4 : 2;          // panels per load batch; two batches are in flight
  using acc_t = typename mma16<T>::acc_t;
  __shared__ acc_t s_acc[kNarrowWaves][NB][64];
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);      // (its panels are counted in scalar registers)
  const int64_t i0 = (int64_t)blockIdx.x * 16;
  const int64_t npanels = k / KSTEP;
  const int nwaves = blockDim.x >> 6;
  const int64_t p_begin = wave * npanels / nwaves, p_end = (wave + 1) * npanels / nwaves;
  const uint8_t* bp[NB];
#pragma unroll
  for (int f = 0; f < NB; f++) {
    const int64_t col = f * 16 + li < n_dense ? f * 16 + li : n_dense - 1;      // clamp: the column is never stored
    bp[f] = b + col * ldb_bytes + lk * 16;
  }
  const uint8_t* av = a_values + (i0 + li) * 64 + lk * 16;
  const uint8_t* am = a_meta + panel_meta_offset(lk * (M_ROW / 4), i0 + li, n_sparse);   // (a panel's further words: n_sparse * 4 bytes apart)
  const int64_t a_step = n_sparse * 64, m_step = n_sparse * M_ROW;
  acc_t acc[NB];                             // (of consecutive instructions, so that none waits for the one before)
#pragma unroll
  for (int f = 0; f < NB; f++)
#pragma unroll
    for (int r = 0; r < 4; r++) acc[f][r] = 0;
  // two register sets: the loads of the next batch are in flight while the current one is multiplied
  int4v af[2][BATCH], lo[2][BATCH][NB], hi[2][BATCH][NB];
  int idx[2][BATCH];
  auto load_batch = [&](int set, int64_t p) {
#pragma unroll
    for (int u = 0; u < BATCH; u++) {
      const int64_t pp = p + u < p_end ? p + u : p_end - 1;     // past the end: re-read the last panel, do not multiply it
      af[set][u] = __builtin_nontemporal_load(reinterpret_cast<const int4v*>(av + pp * a_step));
      if constexpr (sizeof(T) == 2) idx[set][u] = *reinterpret_cast<const uint16_t*>(am + pp * m_step);
      else idx[set][u] = *reinterpret_cast<const int*>(am + pp * m_step);
#pragma unroll
      for (int f = 0; f < NB; f++) {
        lo[set][u][f] = *reinterpret_cast<const int4v*>(bp[f] + pp * 128);
        hi[set][u][f] = *reinterpret_cast<const int4v*>(bp[f] + pp * 128 + 64);
      }
    }
  };
  auto multiply = [&](int set, int u) {
#pragma unroll
    for (int f = 0; f < NB; f++) {
      const int4v l = lo[set][u][f], h = hi[set][u][f];
      const int8v bfrag = {l[0], l[1], l[2], l[3], h[0], h[1], h[2], h[3]};
      acc[f] = mma16<T>::template run<0>(af[set][u], bfrag, acc[f], idx[set][u]);
    }
  };
  // (the scheduling barriers keep the loads ahead of the instructions that wait for the previous batch)
  auto multiply_batch = [&](int set) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < BATCH; u++) multiply(set, u);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto multiply_last = [&](int set, int64_t p) {
#pragma unroll
    for (int u = 0; u < BATCH; u++)
      if (p + u < p_end) multiply(set, u);
  };
  int64_t p = p_begin;
  if (p < p_end) load_batch(0, p);
  for (; p + 2 * BATCH <= p_end; p += 2 * BATCH) {
    load_batch(1, p + BATCH);
    multiply_batch(0);
    if (p + 2 * BATCH < p_end) load_batch(0, p + 2 * BATCH);
    multiply_batch(1);
  }
  if (p + BATCH < p_end) {
    load_batch(1, p + BATCH);
    multiply_batch(0);
    multiply_last(1, p + BATCH);
  } else if (p < p_end) {
    multiply_last(0, p);
  }
#pragma unroll
  for (int f = 0; f < NB; f++) s_acc[wave][f][lane] = acc[f];
  __syncthreads();
  for (int f = wave; f < NB; f += nwaves) {  // a wave finishes every nwaves-th fragment, its pieces added in wave order
    const int64_t col = f * 16 + li;
    if (col >= n_dense) continue;
    acc_t sum = s_acc[0][f][lane];
#pragma unroll
    for (int w = 1; w < nwaves; w++) sum += s_acc[w][f][lane];
    const int64_t row = i0 + lk * 4;         // D layout: column l%16, rows 4*(l/16) + r
    OutT o[4];
#pragma unroll
    for (int r = 0; r < 4; r++) o[r] = to_out<OutT>(finish_value(sum[r], scale, bias, row + r, act));
    if constexpr (C_JMAJOR) {
      *reinterpret_cast<Pack<OutT, 4>*>(c + col * ldc + row) = *reinterpret_cast<Pack<OutT, 4>*>(o);
    } else {
#pragma unroll
      for (int r = 0; r < 4; r++) c[(row + r) * ldc + col] = o[r];
    }
  }
}

// Up to 32 dense columns (NC = 8, 16 or 32): a block owns 16 sparse rows, its NW waves each take a share of the k range and meet in LDS at the
// end (added in wave order).  Bound by the one pass over the compressed operand (50.7 MB of fp16 11008 x 4096, 7.9 us at the rate of a copy) and
// what a launch, its first loads and its last store take beside it (768 x 768: 2.8 us).  A wave keeps two chunks of 8 panels in flight, in
// registers; nothing it loads comes from the dense operand but each of the columns there are once, 1 KB a chunk, handed to the fragments
// through LDS of its own (no barrier: wave_lds_fence).  Read as fragments from memory the dense operand costs
// twice the sparse one's requests, and a compute unit takes 64 bytes of them a clock; shared by the waves of a block, 16 panels between two
// barriers, it leaves a third of the compute units without a block.  The metadata of two panels are one load of a word per lane,
// brought to their lanes by swaps of rows.  Adjacent row blocks, which share the lines of their metadata, are dealt to the same XCD.
// us before and now, fp16, operands from memory, one column: 11008 x 4096 12.5 and 10.6, 8192 x 8192 17.7 and 14.0, 4096 x 11008 12.8 and 11.3,
// 4096 x 4096 6.6 and 5.7, 768 x 3072 5.3 and 4.0; eight: 12.8 and 11.7, 17.8 and 15.8, 14.5 and 12.8, 7.0 and 6.1.  Chunks of
// 16 panels 11008 x 4096 13.6, 8192 x 8192 15.1; two row blocks a wave 12.2 and 15.1 (against 16 columns 14.6 and 16.5, here 14.1 and 19.1).
// 24 columns, before on fragments from memory or on 256 x 64 tiles and two launches: 4096 x 4096 12.7 and 8.5, 4096 x 8192 15.0 and 13.2, 10240 x 2048
// 13.3 and 10.3, 768 x 3072 8.6 and 6.9; two row blocks a wave there 9.9, 20.2, 11.3, 9.3; 64 columns of 4096 x 4096 on four fragments 13.8 for 14.9, but of
// 8192 x 8192 33 for 23.
template <typename T, typename OutT, bool C_JMAJOR, int NC, int NW>
__global__ void __launch_bounds__(64 * NW)
spmm_few(const uint8_t* __restrict__ a_values, const uint8_t* __restrict__ a_meta, int64_t n_sparse, int64_t k,
         const uint8_t* __restrict__ b, int64_t ldb_bytes, int64_t n_dense,
         OutT* __restrict__ c, int64_t ldc, const OutT* __restrict__ bias, float scale, int act) {
  constexpr int KSTEP = mma16<T>::KSTEP;
  constexpr int NB = (NC + 15) / 16, CHAINS = NB == 1 ? 2 : 1;                    // fragments of 16 columns; instructions in a row that do not wait on each other
  constexpr int CH = NB == 1 ? 8 : 4;                 // panels per chunk
  constexpr int COLS = 8 / CH, LOADS = NC / COLS;     // a load of the wave brings 16 bytes a lane, the chunk of COLS dense columns
  constexpr bool PAIR = sizeof(T) == 2;               // two words of metadata per row and panel (8-bit values: four, one for each lane of a row)
  using acc_t = typename mma16<T>::acc_t;
  __shared__ __attribute__((aligned(16))) uint8_t s_b[NW][CH * NC * 128];
  __shared__ acc_t s_acc[NW - 1][NB][64];
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t blocks16 = n_sparse / 16, per_xcd = (blocks16 + 7) / 8;           // (workgroup ids are dealt to the XCDs round-robin)
  const int64_t rb = (int64_t)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((int64_t)(blockIdx.x >> 3) >= per_xcd || rb >= blocks16) return;
  const int64_t i0 = rb * 16, npanels = k / KSTEP;
  const int p_begin = (int)(wave * npanels / NW), p_end = (int)((wave + 1) * npanels / NW);
  const uint8_t* av = a_values + (i0 + li) * 64 + lk * 16;
  const uint8_t* am = a_meta + (i0 + li) * 4;
  const int64_t a_step = n_sparse * 64, word_step = n_sparse * 4;
  // the wave's chunk of the dense operand: [panel][column][128 bytes], the 16-byte pieces of a column XOR-swizzled by column / 2, so that
  // the 16 lanes that read one piece position of 16 columns hit different banks
  uint8_t* const sb = s_b[wave];
  int rd_lo[NB], rd_hi[NB];
  acc_t acc[NB][CHAINS];
#pragma unroll
  for (int f = 0; f < NB; f++) {
    const int col = min(f * 16 + li, (int)n_dense - 1);         // (of a column past the last nothing is stored)
    rd_lo[f] = col * 128 + ((lk ^ ((col >> 1) & 7)) * 16);
    rd_hi[f] = col * 128 + (((lk + 4) ^ ((col >> 1) & 7)) * 16);
#pragma unroll
    for (int h = 0; h < CHAINS; h++)
#pragma unroll
      for (int r = 0; r < 4; r++) acc[f][h][r] = 0;
  }
  const int b_col = lane / (CH * 8), b_panel = lane / 8 % CH, b_piece = lane & 7;
  int4v af[2][CH], breg[LOADS];
  uint32_t words[2][PAIR ? CH / 2 : CH];
  auto load_a = [&](int set, int p) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < CH; u++) {
      const int pp = min(p + u, p_end - 1);           // past the end: re-read the last panel, do not multiply it
      af[set][u] = __builtin_nontemporal_load(reinterpret_cast<const int4v*>(av + pp * a_step));
      if constexpr (!PAIR) words[set][u] = *reinterpret_cast<const uint32_t*>(am + (pp * 4 + lk) * word_step);
      else if (u % 2 == 0) words[set][u / 2] = *reinterpret_cast<const uint32_t*>(am + min((p + u) * 2 + lk, p_end * 2 - 1) * word_step);
    }
  };
  auto load_b = [&](int p) __attribute__((always_inline)) {
    const int64_t at = (int64_t)min(p + b_panel, p_end - 1) * 128 + b_piece * 16;
#pragma unroll
    for (int j = 0; j < LOADS; j++)
      if (j * COLS < n_dense) breg[j] = *reinterpret_cast<const int4v*>(b + (COLS == 1 ? j : min((int64_t)(j * COLS + b_col), n_dense - 1)) * ldb_bytes + at);
  };
  auto store_b = [&]() __attribute__((always_inline)) {
    wave_lds_fence();                                 // behind the reads of the chunk before
#pragma unroll
    for (int j = 0; j < LOADS; j++) {
      const int col = j * COLS + b_col;
      if (j * COLS < n_dense) *reinterpret_cast<int4v*>(sb + (b_panel * NC + col) * 128 + ((b_piece ^ ((col >> 1) & 7)) * 16)) = breg[j];
    }
    wave_lds_fence();
  };
  auto index_of = [&](int set, int u) __attribute__((always_inline)) {
    if constexpr (PAIR) {
      // row r of 16 lanes holds word r of the pair of panels; it needs the half r % 2 of word r / 2 of its panel
      typedef uint32_t uint2v __attribute__((ext_vector_type(2)));
      const uint2v panels = __builtin_amdgcn_permlane32_swap(words[set][u / 2], words[set][u / 2], false, false);      // words 0 1 0 1, and 2 3 2 3
      const uint2v both = __builtin_amdgcn_permlane16_swap(panels[u % 2], panels[u % 2], false, false);                // of it 0 0 0 0, and 1 1 1 1
      return (int)((lk < 2 ? both[0] : both[1]) >> ((lk & 1) * 16));
    } else {
      return (int)words[set][u];
    }
  };
  auto multiply_panel = [&](int set, int u) __attribute__((always_inline)) {
    const int idx = index_of(set, u);
#pragma unroll
    for (int f = 0; f < NB; f++) {
      const int4v lo = *reinterpret_cast<const int4v*>(sb + u * NC * 128 + rd_lo[f]);
      const int4v hi = *reinterpret_cast<const int4v*>(sb + u * NC * 128 + rd_hi[f]);
      const int8v bfrag = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      acc[f][u % CHAINS] = mma16<T>::template run<0>(af[set][u], bfrag, acc[f][u % CHAINS], idx);
    }
  };
  auto multiply = [&](int set, int p) __attribute__((always_inline)) {
    if (p + CH <= p_end) {
#pragma unroll
      for (int u = 0; u < CH; u++) multiply_panel(set, u);
    } else {
#pragma unroll
      for (int u = 0; u < CH; u++)
        if (p + u < p_end) multiply_panel(set, u);
    }
  };
  if (p_begin < p_end) {
    load_b(p_begin);
    load_a(0, p_begin);
    __builtin_amdgcn_sched_barrier(0);                // (the scheduling barriers keep a chunk's loads ahead of the instructions that wait for the one before)
    for (int p = p_begin; p < p_end; p += 2 * CH) {
      store_b();
      if (p + CH < p_end) { load_b(p + CH); load_a(1, p + CH); }
      __builtin_amdgcn_sched_barrier(0);
      multiply(0, p);
      __builtin_amdgcn_sched_barrier(0);
      if (p + CH < p_end) {
        store_b();
        if (p + 2 * CH < p_end) { load_b(p + 2 * CH); load_a(0, p + 2 * CH); }
        __builtin_amdgcn_sched_barrier(0);
        multiply(1, p + CH);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
#pragma unroll
  for (int f = 0; f < NB; f++) {
    if constexpr (CHAINS == 2) acc[f][0] += acc[f][CHAINS - 1];
    if (wave > 0) s_acc[wave - 1][f][lane] = acc[f][0];
  }
  __syncthreads();
  if (wave > 0) return;
  const int64_t row = i0 + lk * 4;           // D layout: column l%16, rows 4*(l/16) + r
#pragma unroll
  for (int f = 0; f < NB; f++) {
    const int64_t col = f * 16 + li;
    if (col >= n_dense) continue;
    acc_t sum = acc[f][0];
#pragma unroll
    for (int w = 1; w < NW; w++) sum += s_acc[w - 1][f][lane];
    OutT o[4];
#pragma unroll
    for (int r = 0; r < 4; r++) o[r] = to_out<OutT>(finish_value(sum[r], scale, bias, row + r, act));
    if constexpr (C_JMAJOR) {
      *reinterpret_cast<Pack<OutT, 4>*>(c + col * ldc + row) = *reinterpret_cast<Pack<OutT, 4>*>(o);
    } else {
#pragma unroll
      for (int r = 0; r < 4; r++) c[(row + r) * ldc + col] = o[r];
    }
  }
}

// Waves that share a row block: some 1400 to 2000 waves in all, and six panels for each of them, or two; from 17 columns on, where a wave's
// chunks are of four panels, so many that one chunk holds a wave's share: a second one, begun for a panel or two, costs half as much again with 16-bit values and
// up to all of it with 8-bit ones.  us in four waves and in eight, 17 panels: fp16 3072 x 1088 against 26 columns 5.7 and 5.0, e4m3 3008 x 2176 against 30 8.7 and 5.3; 20
// panels: e4m3 2912 x 2560 against 31 9.4 and 5.6 (before spmm_few 5.2, 5.3, 6.1).  us with 2, 4 and 8, fp16, one column:
// 11008 x 4096 (688 row blocks) 10.6, 11.0 and 12.7; 8192 x 8192 (512) 14.0, 14.3 and 15.8; 6144 x 4096 (384) 7.9, 7.8 and 8.6;
// 4096 x 11008 (256) 13.9, 11.4 and 11.3; 768 x 3072 (48) 4.7, 4.3 and 4.0; 3072 x 768 (192, 12 panels) 2.96, 3.03 and 3.6.  24 columns:
// 11008 x 1024 6.7, 7.6 and 12.2; 8192 x 2048 9.4, 8.0 and 9.4; 4096 x 2048 8.0, 6.2 and 5.5; 768 x 768 against 32 5.1, 4.2 and 4.9.
inline int few_waves(int64_t blocks, int64_t npanels, int64_t n_dense) {
  const bool many = n_dense > 16;
  int waves = blocks <= 256 ? 8 : many || blocks < 512 ? 4 : 2;
  while (waves > 2 && (many ? npanels <= 2 * waves : npanels < 6 * waves)) waves /= 2;
  return waves;
}

// Up to how many dense columns the narrow kernels are the faster ones; of 200 products, us narrow and on 128 x 64 tiles (float16 if not said otherwise):
// 9 to 16 on spmm_few up to 128 panels (16 columns of 5120 x 1280 6.0 and 7.2, of 2560 x 2304 6.0 and 7.9, of 4096 x 4096 e4m3 7.3 and 9.7, of
// 3168 x 5504 9.3 and 10.0), 72 where fewer than 96 row blocks leave compute units without one (of 1888 x 4352 7.3 and 8.4, but of 736 x 5120 8.7 and 8.1), and some
// further with neither many nor few (of 4096 x 11008 14.6 and 14.8).
// 17 to 32, whose fragments cost requests with every panel of every block, up to 64 panels and one block to a compute unit (24 of 4096 x 4096 8.6 and
// 9.5, 32 of 4096 x 1792 5.6 and 8.7, of 1024 x 4096 7.9 and 7.7; with more panels 24 of 1600 x 6400 10.9 and 8.9, 32 of 4096 x 8192 14.7 and 13.1), with
// two blocks 32 panels, of 8-bit values, which have twice the metadata, 16, and up to 24 columns 32 of them on spmm_narrow (24 of 6048 x 2112 8.6 and 9.3, 32 of
// 5120 x 1280 7.6 and 7.3, but of 6144 x 4096 13.5 and 10.8; e4m3 19 of 7520 x 3840 8.9 and 11.6, 20 of 6496 x 3072 8.6 and 9.7, but 30 of 5728 x 2432 8.4 and 7.7);
// with more blocks none (32 of 9824 x 448 6.0 and 5.0, of 14688 x 1856 12.5 and 9.1).
// 33 to 48 on spmm_narrow up to 24 panels and one block (40 of 2304 x 768 4.9 and 5.7, 48 of 960 x 1472 7.5 and 7.7, but of 4320 x 1216 11.1 and 7.1); to 64 up
// to nine panels (64 of 1088 x 320 5.1 and 5.0, but of 2304 x 768 6.0 and 5.8, of 3840 x 1280 9.1 and 7.4).  A weight of less than 64 rows takes no tiles.
inline int64_t narrow_columns(int64_t n_sparse, int64_t npanels, bool eight_bit) {
  const int64_t blocks = n_sparse / 16;
  if (blocks <= 256 && npanels <= 24) return npanels <= 9 || n_sparse < 64 ? 64 : 48;
  if (npanels <= (blocks <= 256 ? 64 : blocks > 512 ? 0 : eight_bit ? 16 : 32)) return 32;
  if (eight_bit && blocks <= 512 && npanels <= 32) return 24;
  if (npanels <= (blocks < 96 ? 72 : blocks <= 256 ? 192 : 128)) return 16;
  return blocks >= 512 ? 10 : 8;
}

// Whether so many columns (up to narrow_columns) take spmm_few.  9 to 16 of a short k do not with up to two blocks a compute unit: a wave
// has its dense columns brought in whole chunks of 8 panels, 16 loads of which most are of no use.  us before spmm_few, on it, and on
// spmm_narrow again, 16 columns: fp16 256 x 256 (4 panels) 2.88, 3.36, 2.88, 2144 x 256 3.13, 3.42, 3.13; e4m3 864 x 384 3.04, 3.42, 3.04; with two blocks a unit
// from memory alike (6016 x 256 3.7), from the caches 3.3, 3.7, 3.3; with more spmm_few is the faster one by a fifth, with 8 panels
// as fast (3.2).  17 to 32: from kFewPanels panels on, of 8-bit values against more than one
// block a compute unit, whose share of a wave is then more than one chunk, up to 16 (24 columns of e4m3 5696 x 2816 9.2, on spmm_narrow 8.6).
constexpr int64_t kShortPanels = 8;
inline bool takes_few(int64_t blocks, int64_t npanels, int64_t n_dense, bool eight_bit) {
  if (n_dense <= 16) return n_dense <= 8 || blocks > 512 || npanels >= kShortPanels;
  return n_dense <= 32 && npanels >= kFewPanels && !(eight_bit && blocks > 256 && npanels > 16);
}

template <typename T, typename OutT>
int launch_narrow(const void* av, const void* am, int64_t n_sparse, int64_t k, const void* b, int64_t ldb, int64_t n_dense,
                  void* c, int c_layout, int64_t ldc, const void* bias, float scale, int act, hipStream_t s) {
  dim3 grid((unsigned)(n_sparse / 16));
  const int64_t blocks = n_sparse / 16, npanels = k * (int64_t)sizeof(T) / 128;
  if (takes_few(blocks, npanels, n_dense, sizeof(T) == 1)) {
    const int nw = few_waves(blocks, npanels, n_dense);
    auto go = [&](auto jmajor, auto nc, auto nwc) {
      hipLaunchKernelGGL((spmm_few<T, OutT, decltype(jmajor)::value, decltype(nc)::value, decltype(nwc)::value>), dim3((unsigned)((blocks + 7) / 8 * 8)),
                         dim3(64 * decltype(nwc)::value), 0, s,
                         (const uint8_t*)av, (const uint8_t*)am, n_sparse, k, (const uint8_t*)b, ldb * (int64_t)sizeof(T), n_dense,
                         (OutT*)c, ldc, (const OutT*)bias, scale, act);
    };
    auto go_nw = [&](auto jmajor, auto nc) {
      if (nw == 8) go(jmajor, nc, std::integral_constant<int, 8>{});
      else if (nw == 4) go(jmajor, nc, std::integral_constant<int, 4>{});
      else go(jmajor, nc, std::integral_constant<int, 2>{});
    };
    auto go_nc = [&](auto jmajor) {
      if (n_dense <= 8) go_nw(jmajor, std::integral_constant<int, 8>{});
      else if (n_dense <= 16) go_nw(jmajor, std::integral_constant<int, 16>{});
      else go_nw(jmajor, std::integral_constant<int, 32>{});
    };
    if (c_layout == TF24_COL_MAJOR) go_nc(std::true_type{}); else go_nc(std::false_type{});
    return check_launch("tf24_spmm");
  }
  int nwaves = kNarrowWaves;                                    // few row blocks: the waves of a block split k
  while (nwaves > 1 && npanels / nwaves < 4) nwaves /= 2;
  auto go = [&](auto jmajor, auto nb) {
    hipLaunchKernelGGL((spmm_narrow<T, OutT, decltype(jmajor)::value, decltype(nb)::value>), grid, dim3(64 * nwaves), 0, s, (const uint8_t*)av,
                       (const uint8_t*)am, n_sparse, k, (const uint8_t*)b, ldb * (int64_t)sizeof(T), n_dense, (OutT*)c, ldc, (const OutT*)bias, scale, act);
  };
  auto go_nb = [&](auto jmajor) {
    if (n_dense <= 16) go(jmajor, std::integral_constant<int, 1>{});
    else if (n_dense <= 32) go(jmajor, std::integral_constant<int, 2>{});
    else if (n_dense <= 48) go(jmajor, std::integral_constant<int, 3>{});
    else go(jmajor, std::integral_constant<int, 4>{});
  };
  if (c_layout == TF24_COL_MAJOR) go_nb(std::true_type{}); else go_nb(std::false_type{});
  return check_launch("tf24_spmm");
}

template <typename T, typename OutT>
int launch_general(const void* av, const void* am, int a_layout, int64_t n_sparse, int64_t k, const void* b, int b_layout, int64_t ldb,
                   int64_t n_dense, void* c, int c_layout, int64_t ldc, const void* bias, float scale, int act, hipStream_t s) {
  dim3 grid((unsigned)((n_dense + 63) / 64), (unsigned)((n_sparse + 63) / 64));
  const bool kc = b_layout == TF24_ROW_MAJOR, jm = c_layout == TF24_COL_MAJOR;
#define TF24_GO(KC, JM)                                                                                              \
  hipLaunchKernelGGL((spmm_general<T, OutT, KC, JM>), grid, dim3(256), 0, s, (const uint8_t*)av, (const uint8_t*)am, \
                     n_sparse, k, (const T*)b, ldb, n_dense, (OutT*)c, ldc, (const OutT*)bias, scale, act, a_layout)
  if (kc && jm) TF24_GO(true, true);
  else if (kc) TF24_GO(true, false);
  else if (jm) TF24_GO(false, true);
  else TF24_GO(false, false);
#undef TF24_GO
  return check_launch("tf24_spmm");
}

template <typename T>
int dispatch_out(int out_dtype, const void* av, const void* am, int a_layout, int64_t n_sparse, int64_t k, const void* b, int b_layout,
                 int64_t ldb, int64_t n_dense, void* c, int c_layout, int64_t ldc, const void* bias, float scale, int act,
                 void* workspace, int64_t workspace_bytes, hipStream_t s, RowSums* sums) {
  const bool panel = a_layout == TF24_COMPRESSED_PANEL;
  // the tiled kernel reads a k-strided dense operand through transposing LDS reads (16-bit types only)
  // (also for a narrow dense operand: with its k pieces the tiled kernel beats the general one from 8 columns on)
  const bool tiled = panel && (b_layout == TF24_ROW_MAJOR || sizeof(T) == 2) && n_sparse >= 64;
  // up to 64 dense columns: the tiled kernel on 128 x 64 tiles (or 256 x 64: takes_tall_slim); more: 128 x 128 (takes_small), 192 x 128 (takes_lower), 256 x 128 or 256 x 256 tiles (takes_mid)
  const bool slim = tiled && b_layout == TF24_ROW_MAJOR && n_dense <= SlimCfg::BJ;
  const bool tall_slim = slim && takes_tall_slim(n_sparse, k * (int64_t)sizeof(T) / SlimCfg::KB, sizeof(T) == 1);
  const bool small = tiled && b_layout == TF24_ROW_MAJOR && takes_small<T>(n_sparse, k, n_dense, workspace ? workspace_bytes : 0);
  const bool lower = tiled && b_layout == TF24_ROW_MAJOR && takes_lower<T>(n_sparse, k, n_dense, workspace ? workspace_bytes : 0);
  const bool mid = tiled && b_layout == TF24_ROW_MAJOR && takes_mid<T>(n_sparse, k, n_dense, workspace ? workspace_bytes : 0);
  // few dense columns: one pass over the compressed operand (narrow_columns), also up to 16 when the tiled kernel cannot cut k
  // into pieces (no workspace), which it needs to fill the chip
  const bool narrow = panel && b_layout == TF24_ROW_MAJOR &&
                      (n_dense <= narrow_columns(n_sparse, k * (int64_t)sizeof(T) / 128, sizeof(T) == 1) || (n_dense <= 16 && !(slim && workspace)));
  if constexpr (std::is_same<T, i8_t>::value) {        // integer product: int32 accumulators, results and bias
    if (narrow) return launch_narrow<T, int32_t>(av, am, n_sparse, k, b, ldb, n_dense, c, c_layout, ldc, bias, scale, act, s);
    if (tall_slim) return launch_tiled<T, int32_t, TallSlimCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
    if (slim) return launch_tiled<T, int32_t, SlimCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
    if (small) return launch_tiled<T, int32_t, SmallCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
    if (lower) return launch_tiled<T, int32_t, LowerCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
    if (mid) return launch_tiled<T, int32_t, MidCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
    if (tiled) return launch_tiled<T, int32_t, TiledCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
    return launch_general<T, int32_t>(av, am, a_layout, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, s);
  } else {
  if (narrow) {
    switch (out_dtype) {
      case TF24_F16: return launch_narrow<T, f16_t>(av, am, n_sparse, k, b, ldb, n_dense, c, c_layout, ldc, bias, scale, act, s);
      case TF24_BF16: return launch_narrow<T, bf16_t>(av, am, n_sparse, k, b, ldb, n_dense, c, c_layout, ldc, bias, scale, act, s);
      case TF24_F32: return launch_narrow<T, float>(av, am, n_sparse, k, b, ldb, n_dense, c, c_layout, ldc, bias, scale, act, s);
    }
  }
  if (tall_slim) {
    switch (out_dtype) {
      case TF24_F16: return launch_tiled<T, f16_t, TallSlimCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
      case TF24_BF16: return launch_tiled<T, bf16_t, TallSlimCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
      case TF24_F32: return launch_tiled<T, float, TallSlimCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
    }
  }
  if (slim) {
    switch (out_dtype) {
      case TF24_F16: return launch_tiled<T, f16_t, SlimCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
      case TF24_BF16: return launch_tiled<T, bf16_t, SlimCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
      case TF24_F32: return launch_tiled<T, float, SlimCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
    }
  }
  if (small) {
    switch (out_dtype) {
      case TF24_F16: return launch_tiled<T, f16_t, SmallCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
      case TF24_BF16: return launch_tiled<T, bf16_t, SmallCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
      case TF24_F32: return launch_tiled<T, float, SmallCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
    }
  }
  if (lower) {
    switch (out_dtype) {
      case TF24_F16: return launch_tiled<T, f16_t, LowerCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
      case TF24_BF16: return launch_tiled<T, bf16_t, LowerCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
      case TF24_F32: return launch_tiled<T, float, LowerCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
    }
  }
  if (mid) {
    switch (out_dtype) {
      case TF24_F16: return launch_tiled<T, f16_t, MidCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
      case TF24_BF16: return launch_tiled<T, bf16_t, MidCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
      case TF24_F32: return launch_tiled<T, float, MidCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s);
    }
  }
  if (tiled) {
    switch (out_dtype) {
      case TF24_F16: return launch_tiled<T, f16_t, TiledCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s, sums);
      case TF24_BF16: return launch_tiled<T, bf16_t, TiledCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s, sums);
      case TF24_F32: return launch_tiled<T, float, TiledCfg>(av, am, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s, sums);
    }
  }
  switch (out_dtype) {
    case TF24_F16: return launch_general<T, f16_t>(av, am, a_layout, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, s);
    case TF24_BF16: return launch_general<T, bf16_t>(av, am, a_layout, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, s);
    case TF24_F32: return launch_general<T, float>(av, am, a_layout, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, s);
  }
  return fail(TF24_ERR_DTYPE, "tf24_spmm: unsupported output dtype %d", out_dtype);
  }
}

}  // namespace

// One translation unit per operand type instantiates the kernels of that type (spmm_<type>.hip) behind
// one of these functions; tf24_spmm (spmm.hip) validates and dispatches on the type.  `sums`: row sums that the product's last launch may
// finish as well; it clears their `partial` if it does.
#define TF24_SPMM_ENTRY_ARGS int out_dtype, const void* av, const void* am, int a_layout, int64_t n_sparse, int64_t k, const void* b, int b_layout, \
                 int64_t ldb, int64_t n_dense, void* c, int c_layout, int64_t ldc, const void* bias, float scale, int act, \
                 void* workspace, int64_t workspace_bytes, hipStream_t s, RowSums* sums
#define TF24_SPMM_ENTRY_PASS out_dtype, av, am, a_layout, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, act, workspace, workspace_bytes, s, sums
int spmm_f16(TF24_SPMM_ENTRY_ARGS);
int spmm_bf16(TF24_SPMM_ENTRY_ARGS);
int spmm_e4m3(TF24_SPMM_ENTRY_ARGS);
int spmm_e5m2(TF24_SPMM_ENTRY_ARGS);
int spmm_i8(TF24_SPMM_ENTRY_ARGS);
}  // namespace tf24
