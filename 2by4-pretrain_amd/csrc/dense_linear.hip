// Products of a layer whose weight is dense, 16-bit operands, float32 accumulation, one rounding:
//
//     Y[t, i] = sum_k X[t, k] * W(i, k) + bias[i]
//
// X [tokens, k] row-major.  W(i, k) lies at i * ldw + k (the forward product) or, STRIDED, at k * ldw + i (the gradient of the
// input, whose summed axis is the slow one of the weight).
//
// A block of four waves (2 x 2, one per SIMD) computes 192(i) x 192(t) tiles, wave tile 96 x 96 = 6 x 6 V_MFMA_F32_16X16X32 with 144
// accumulators.  64 elements of k of both operands are one stage of 48 KB, three of which rotate through the LDS: while stage s is
// multiplied, the copies of s + 1 and s + 2 are in flight (global -> LDS directly).  The fragments of a step of 32 elements of k are
// read behind the matrix instructions of the step before, one read behind each.  One workgroup per compute unit walks the tiles of its
// XCD in one pipeline: the copies of the next tile's first two stages ride in the last two stages of the current one, and the
// output pass stages through the buffer that is free.
//
// Bound by the power that the matrix cores may draw: a stage takes 0.53 us on operands of zeros (0.48 by matrix instructions alone) and 0.87
// on random ones, and a launch 8 us beside its stages.  Hence the 16 x 16 instructions: alone, on random operands in registers, they sustain
// 1.9 PFLOP/s where the 32 x 32 ones do 1.65 (2.46 and 2.48 on zeros), and the products below took 1 to 5 % longer with the latter.
// 12288 tokens, bf16, here and in the library (GPU time): 3072 x 768 with bias 57.9 and 62.8 us, 768 x 3072 49 and 63, their input
// gradients 49.5 and 61, 58.8 and 72.  The reads of a step spread over its instructions or over the
// first two thirds of them: alike.  Ordinary instead of streaming stores: 67 us for 61 (3072 x 768).
#include "lds_copies.hpp"
#include <algorithm>
#include <type_traits>

namespace tf24 {
namespace {

typedef short short8v __attribute__((ext_vector_type(8)));

constexpr int kTile = 192, kThreads = 256, kWaves = 4, kFrags = 6;          // fragments of 16 rows (and of 16 columns) per wave
constexpr int kStageK = 64, kRowBytes = kStageK * 2, kStridedRowBytes = kTile * 2;
constexpr int kOperand = kTile * kRowBytes, kStage = 2 * kOperand;          // [W | X]
constexpr int kCopies = kOperand / 1024 / kWaves;                           // 1 KB copies per wave and operand of a stage
// from so many stages on the tiles of XCD x take them from the x-th eighth of k on and wrap round: all XCDs at the same stage read the
// same few memory channels (a stage is 128 bytes from each row, rows lie some 4 KB apart).  us without and with: 1024 x 4096 against
// 6912 57.8 and 54.7, 1280 x 5120 against 4416 66.5 and 62.2, 1600 x 6400 against 2831 71 and 68; 48 stages alike
constexpr int kRotateMinStages = 24;
static_assert(kRotateMinStages - 2 - (7 * kRotateMinStages >> 3) >= 1, "the first three stages of a tile are copied before the order wraps");
constexpr int kRaster = 8;                                                  // tiles along i of a group

__device__ __forceinline__ float4v mma(f16_t, int4v a, int4v b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
}
__device__ __forceinline__ float4v mma(bf16_t, int4v a, int4v b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

template <typename T, bool STRIDED>
__global__ void __launch_bounds__(kThreads)
dense_linear(const uint8_t* __restrict__ w, int64_t ldw, const uint8_t* __restrict__ x, int64_t ldx, int64_t rows, int64_t k, int64_t tokens,
             T* __restrict__ y, int64_t ldy, const T* __restrict__ bias, int tiles_i, int tiles_j, int stagger_ticks) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[3 * kStage];
  // workgroup ids are dealt to the 8 XCDs round-robin: each XCD takes a run of tiles in a raster of groups of kRaster rows of tiles,
  // its workgroup number s the s-th of them and every `slots`-th after it
  const int ntiles = tiles_i * tiles_j, per_xcd = (ntiles + 7) / 8, slots = (int)(gridDim.x >> 3);
  const int xcd = (int)(blockIdx.x & 7), slot = (int)(blockIdx.x >> 3), xcd_end = min((xcd + 1) * per_xcd, ntiles);
  int tile = xcd * per_xcd + slot;
  if (tile >= xcd_end) return;
  int group = __builtin_amdgcn_readfirstlane(tile / (kRaster * tiles_j)), in_group = tile - group * (kRaster * tiles_j);
  auto locate = [&](int64_t& ti0, int64_t& tj0) {                // origin of the tile number in_group of the group
    const int gh = min(kRaster, tiles_i - group * kRaster);
    int col = (unsigned)in_group / kRaster;
    if (gh != kRaster) col = __builtin_amdgcn_readfirstlane((unsigned)in_group / (unsigned)gh);
    ti0 = (int64_t)(group * kRaster + (in_group - col * gh)) * kTile;
    tj0 = (int64_t)col * kTile;
  };
  auto advance = [&]() {                                         // to the workgroup's next tile
    in_group += slots;
    for (int size = min(kRaster, tiles_i - group * kRaster) * tiles_j; in_group >= size; size = min(kRaster, tiles_i - group * kRaster) * tiles_j) {
      in_group -= size;
      group++;
    }
  };
  int64_t i0, j0;
  locate(i0, j0);
  // every second workgroup of an XCD starts 3 us late, so that not all of them write their tiles out at the same moment (bounded, also
  // in iterations): 4096 x 1024 against 6912 tokens 69.9 -> 64.2 us, 3072 x 768 against 12288 61.4 -> 60.9; 6 us late 66.6, 61.8
  if (stagger_ticks > 0 && (slot & 1)) {
    const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
    for (int spin = 0; spin < 1024 && __builtin_amdgcn_s_memrealtime() - t0 < (uint64_t)stagger_ticks; spin++) __builtin_amdgcn_s_sleep(4);
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wi = wave >> 1, wj = wave & 1, l16 = lane & 15, lq = lane >> 4;
  const int nstages = (int)(k / kStageK);                        // (at least 4)
  const int64_t w_step = STRIDED ? kStageK * ldw : kRowBytes;
  const int first_stage = nstages >= kRotateMinStages ? xcd * nstages >> 3 : 0;

  // ---- copies: number q of a wave brings 1 KB of an operand's stage, 8 rows of 128 bytes with their 16-byte chunks XOR-swizzled by row,
  // or (STRIDED) 1 KB of 64 rows of 384, swizzled for the transposing reads below.  Rows past the operand's last re-read it (or the
  // last chunk of a row), and what is computed from them is not stored.
  auto strided_swizzle = [](uint32_t krow) { return (((krow >> 1) & 1) << 2) | (((krow >> 3) & 1) << 1); };
  uint32_t ow[kCopies], ox[kCopies];
  const uint8_t *w_at, *x_at;
  bool lanes_whole = false;
  auto point_at = [&](int64_t ti0, int64_t tj0) {                // sources of the first stage of the tile at (ti0, tj0)
    const int64_t last_i = rows - 1 - ti0, last_j = tokens - 1 - tj0;
    w_at = (STRIDED ? w : w + ti0 * ldw) + first_stage * w_step;
    x_at = x + tj0 * ldx + first_stage * kRowBytes;
    if constexpr (STRIDED) w_at += ti0 * 2;
    // the lanes' offsets are those of any other tile unless rows of one of the two are clamped
    const bool whole = last_i >= kTile - 1 && last_j >= kTile - 1;
    if (whole && lanes_whole) return;
    lanes_whole = whole;
#pragma unroll
    for (int q = 0; q < kCopies; q++) {
      const int row = (wave * kCopies + q) * 8 + (lane >> 3), chunk = (lane & 7) ^ ((row >> 1) & 7);
      ox[q] = (uint32_t)(min((int64_t)row, last_j) * ldx + chunk * 16);
      if constexpr (STRIDED) {
        const uint32_t piece = (uint32_t)((wave * kCopies + q) * 64 + lane), krow = piece / (kTile / 8);
        const int64_t col = min((int64_t)((piece % (kTile / 8)) ^ strided_swizzle(krow)) * 8, rows - 8 - ti0);
        ow[q] = (uint32_t)(krow * ldw + col * 2);                // (a tile's columns begin before the last eight: rows is a multiple of 8)
      } else {
        ow[q] = (uint32_t)(min((int64_t)row, last_i) * ldw + chunk * 16);
      }
    }
  };
  point_at(i0, j0);
  const uint32_t smem_at = lds_offset(smem);
  auto copy_one = [&](int q, uint32_t buf) {                     // the wave's copies of X, then those of W
    if (q < kCopies) g2l16(x_at, ox[q], smem_at + buf + kOperand + (uint32_t)(wave * kCopies + q) * 1024);
    else g2l16(w_at, ow[q - kCopies], smem_at + buf + (uint32_t)(wave * kCopies + q - kCopies) * 1024);
  };
  auto next_stage = [&]() { w_at += w_step; x_at += kRowBytes; };
  auto copy_stage = [&](uint32_t buf) {
#pragma unroll
    for (int q = 0; q < 2 * kCopies; q++) copy_one(q, buf);
    next_stage();
  };

  float4v acc[kFrags][kFrags];
  auto clear = [&]() {
#pragma unroll
    for (int ti = 0; ti < kFrags; ti++)
#pragma unroll
      for (int tj = 0; tj < kFrags; tj++) acc[ti][tj] = float4v{0, 0, 0, 0};
  };
  clear();

  // ---- fragments of a step (32 elements of k): lane l takes row l % 16, elements 8 * (l / 16) .. + 7.  STRIDED: in a group of 16 lanes,
  // lane i receives the halfwords i % 4 of the source lanes 4e + i / 4 (e = 0..3), so source lane s addresses k-row s / 4 (of
  // four), columns 4 * (s % 4).. of the group's 16; two such reads make eight elements of k.
  const int swizzle = (l16 >> 1) & 7;
  uint32_t a_off[2], b_off[2], t_off[kFrags];
#pragma unroll
  for (int step = 0; step < 2; step++) {
    const uint32_t chunk = (uint32_t)((step * 4 + lq) ^ swizzle) * 16;
    a_off[step] = (uint32_t)(wi * 96 + l16) * kRowBytes + chunk;
    b_off[step] = kOperand + (uint32_t)(wj * 96 + l16) * kRowBytes + chunk;
  }
  if constexpr (STRIDED) {
    const uint32_t krow = lq * 8 + (l16 >> 2);
#pragma unroll
    for (int f = 0; f < kFrags; f++) {
      const uint32_t col = (uint32_t)(wi * 96 + f * 16) + (l16 & 3) * 4;
      t_off[f] = krow * kStridedRowBytes + (((col >> 3) ^ strided_swizzle(krow)) * 16) + ((col >> 2) & 1) * 8;
    }
  }
  int4v af[2][kFrags], bf[2][kFrags];                            // [register set][fragment]
  short4v aq[2][kFrags][2];                                      // STRIDED: the halves of a fragment
  constexpr int A_READS = STRIDED ? 2 * kFrags : kFrags, READS = A_READS + kFrags, MMAS = kFrags * kFrags;
  // the reads of a step in the order the next step's instructions need them: W's first fragment, X's, W's others
  auto read_w = [&](int set, int q, uint32_t buf, int step) {
    if constexpr (STRIDED)
      aq[set][q >> 1][q & 1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_short4_ptr)(lds_ptr_t)(smem + buf + t_off[q >> 1] + (step * 32 + (q & 1) * 4) * kStridedRowBytes));
    else af[set][q] = *reinterpret_cast<const int4v*>(smem + buf + a_off[step] + q * 16 * kRowBytes);
  };
  auto read_one = [&](int set, int n, uint32_t buf, int step) {
    constexpr int FIRST = A_READS / kFrags;
    if (n >= FIRST && n < FIRST + kFrags) bf[set][n - FIRST] = *reinterpret_cast<const int4v*>(smem + buf + b_off[step] + (n - FIRST) * 16 * kRowBytes);
    else read_w(set, n < FIRST ? n : n - kFrags, buf, step);
  };
  auto w_fragment = [&](int set, int f) {
    if constexpr (STRIDED) return __builtin_bit_cast(int4v, __builtin_shufflevector(aq[set][f][0], aq[set][f][1], 0, 1, 2, 3, 4, 5, 6, 7));
    else return af[set][f];
  };
  // The instructions of a step from one register set; behind them, one by one, the next step's reads into the other set and the copies
  // of half a stage.
  auto mma_step = [&](int set, int half, bool copies, uint32_t dst, bool reads, uint32_t src, int rstep) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < MMAS; n++) {
      const int ti = n / kFrags, tj = n % kFrags;
      acc[ti][tj] = mma(T{}, w_fragment(set, ti), bf[set][tj], acc[ti][tj]);
      __builtin_amdgcn_sched_barrier(0);
      if (reads) {
#pragma unroll
        for (int q = n * READS / MMAS; q < (n + 1) * READS / MMAS; q++) read_one(set ^ 1, q, src, rstep);
      }
      if (copies) {
#pragma unroll
        for (int q = 0; q < kCopies; q++)
          if (q * MMAS / kCopies == n) copy_one(half * kCopies + q, dst);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // every wave has its copies of the stage in LDS (`more`: those of the one behind may still fly) and its reads of the stage before done
  auto stage_barrier = [&](bool more) {
    if (more) wait_copies_and_barrier<2 * kCopies, true>();
    else wait_copies_and_barrier<0, true>();
  };

  copy_stage(0);
  copy_stage(kStage);
  uint32_t cur = 0, nxt = kStage, fre = 2 * kStage;              // buffers of stage st, st + 1 and st + 2 (= st - 1)
  auto rotate = [&]() { const uint32_t t = cur; cur = nxt; nxt = fre; fre = t; };
  bool chained = false;                                          // this tile's first two stages were copied under the previous one
  for (;;) {
    // (a chained tile's first two stages were waited for before the previous output pass's first store, so its first two barriers only
    // publish them; from the third on loads complete in order, and the copies issued since are more than the wait allows)
    if (chained) wait_reads_and_barrier();
    else stage_barrier(true);
#pragma unroll
    for (int n = 0; n < READS; n++) read_one(0, n, cur, 0);
#pragma unroll
    for (int q = 0; q < kCopies; q++) copy_one(q, fre);
    mma_step(0, 1, true, fre, true, cur, 1);
    next_stage();
    if (chained) wait_reads_and_barrier();
    else stage_barrier(true);
    // Up to the wrap of the stage order, to the last two stages, and, where a tile follows, through those, whose copies are its first two.
    // (One loop, and few instructions between tiles, which nothing covers: us with stages of their own, in which every copy
    // stood behind a branch, and new offsets and divisions for every tile, and now: 2048 x 512 against 16384 tokens 43.7 and 42.5, 4096 x 1024 against
    // 6912 66.0 and 64.3, 5120 x 1280 against 4416 62.0 and 60.3, 3072 x 768 against 12288 59.7 and 58.9.)
    int st = 1;
    bool has_next = false;
    int64_t next_i0 = i0, next_j0 = j0;
    for (int lim = nstages - 2 - first_stage;;) {
      for (; st < lim; st++) {
        rotate();
        mma_step(1, 0, true, fre, true, cur, 0);                 // the last step of stage st - 1
        mma_step(0, 1, true, fre, true, cur, 1);
        next_stage();
        stage_barrier(true);
      }
      if (st < nstages - 2) {
        w_at -= nstages * w_step;                                // the stage order wraps
        x_at -= nstages * kRowBytes;
        lim = nstages - 2;
        continue;
      }
      if (st >= nstages || tile + slots >= xcd_end) break;
      tile += slots;
      has_next = true;
      advance();
      locate(next_i0, next_j0);
      point_at(next_i0, next_j0);
      lim = nstages;
    }
    for (; st < nstages; st++) {                                 // the last stages of the last tile
      rotate();
      mma_step(1, 0, false, 0, true, cur, 0);
      mma_step(0, 1, false, 0, true, cur, 1);
      stage_barrier(false);
    }
    // the bias of the wave's 96 rows, fetched ahead of the last step
    uint32_t bias_w[2] = {0, 0};
    if (bias) {
#pragma unroll
      for (int q = 0; q < 2; q++) bias_w[q] = reinterpret_cast<const uint16_t*>(bias)[min(i0 + wi * 96 + q * 64 + lane, rows - 1)];
    }
    mma_step(1, 0, false, 0, false, 0, 0);
#pragma unroll
    for (int q = 0; q < 2; q++) asm volatile("" : "+v"(bias_w[q]));

    // ---- output pass: a lane holds column l % 16 and rows 4 * (l / 16) + r of a fragment.  Each wave stages 32(t) x 96(i)
    // pieces in a slice of the last stage's buffer (rows of 192 bytes, chunks XOR-swizzled with the row) and stores whole rows of them.
    constexpr int SLICE = 32 * 192;
    float* bias_lds = reinterpret_cast<float*>(smem + cur + kWaves * SLICE + wave * 384);
#pragma unroll
    for (int q = 0; q < 2; q++)
      if (q * 64 + lane < 96) bias_lds[q * 64 + lane] = to_float(T{(uint16_t)bias_w[q]});
    wave_lds_fence();
    uint8_t* stage = smem + cur + wave * SLICE;
    auto chunk_at = [](int row, int ch) { return row * 192 + (ch ^ ((row >> 2) & 3)) * 16; };
#pragma unroll
    for (int tp = 0; tp < kFrags / 2; tp++) {                    // 32 columns (t)
      if (tp > 0) wave_lds_fence();                              // behind the reads of the piece before
#pragma unroll
      for (int ti = 0; ti < kFrags; ti++) {
        const float4v add = *reinterpret_cast<const float4v*>(bias_lds + ti * 16 + lq * 4);
#pragma unroll
        for (int t2 = 0; t2 < 2; t2++) {
          T o[4];
#pragma unroll
          for (int r = 0; r < 4; r++) o[r] = from_float<T>(acc[ti][tp * 2 + t2][r] + add[r]);
          *reinterpret_cast<Pack<T, 4>*>(stage + chunk_at(t2 * 16 + l16, ti * 2 + (lq >> 1)) + (lq & 1) * 8) = *reinterpret_cast<Pack<T, 4>*>(o);
        }
      }
      if (tp == 0 && has_next) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the next tile's first two stages
      wave_lds_fence();
#pragma unroll
      for (int it = 0; it < 6; it++) {
        const uint32_t piece = it * 64 + lane;
        const int jl = piece / 12, ch = piece % 12;
        const int64_t icol = i0 + wi * 96 + ch * 8, jrow = j0 + wj * 96 + tp * 32 + jl;
        const int4v v = *reinterpret_cast<const int4v*>(stage + chunk_at(jl, ch));
        if (jrow < tokens && icol < rows) __builtin_nontemporal_store(v, reinterpret_cast<int4v*>(y + jrow * ldy + icol));
      }
    }
    if (!has_next) break;
    i0 = next_i0; j0 = next_j0; chained = true;
    rotate();
    clear();
  }
}

template <typename T>
int launch_linear(const void* w, int64_t ldw, bool strided, const void* x, int64_t ldx, int64_t rows, int64_t k, int64_t tokens, void* y, int64_t ldy,
                  const void* bias, hipStream_t s) {
  const int tiles_i = (int)((rows + kTile - 1) / kTile), tiles_j = (int)((tokens + kTile - 1) / kTile);
  const int slots = std::max(1, compute_units() / 8), per_xcd = (tiles_i * tiles_j + 7) / 8;
  const int stagger = per_xcd > slots && k / kStageK <= 32 ? 300 : 0;
  auto go = [&](auto is_strided) {
    hipLaunchKernelGGL((dense_linear<T, decltype(is_strided)::value>), dim3((unsigned)(std::min(per_xcd, slots) * 8)), dim3(kThreads), 0, s, (const uint8_t*)w,
                       ldw * 2, (const uint8_t*)x, ldx * 2, rows, k, tokens, (T*)y, ldy, (const T*)bias, tiles_i, tiles_j, stagger);
  };
  if (strided) go(std::true_type{}); else go(std::false_type{});
  return check_launch("tf24_linear16");
}

// Where the kernel is the faster one, against the library's product (hipBLASLt through torch, GPU time): tiles that fill the rounds of
// the compute units.  `fill` is the share of the rounds' results that the product has.  Of 480 products of S-STE layers (512 to 1600
// wide and four times that, 500 to 16384 tokens, both directions, operands that change from call to call) the rule takes 86: 15 % less
// time than the library over them, 40 % at best, and 2 % more at worst.  fill, library and here, us: 3072 x 768 against 12288
// tokens 1.00 60.1 56.3, its input gradient (768 rows, k 3072, STRIDED) 59.7 48.0; 2560 x 640 against 13317 0.90 58.6 44.8, 5120 x 1280
// against 1074 0.58 22.9 20.2.  Left to the library: several rounds below 0.89 (4096 x 1024 against 4053 0.88 29.0 35.3, 6400 x 1600
// against 2525 0.86 40.2 51.9), one round of long tiles below 0.72 (1600 x 6400 against 2831 0.48 62.5 77.5), where its smaller tiles and its
// pieces of k reach more compute units, and one round of short ones below 0.55 (4096 x 1024 against 1256 0.545 15.2 16.4).
bool suits(int64_t rows, int64_t k, int64_t tokens, int cus) {
  const int64_t tiles = (rows + kTile - 1) / kTile * ((tokens + kTile - 1) / kTile), rounds = (tiles + cus - 1) / cus;
  const double fill = (double)rows * (double)tokens / ((double)(rounds * cus) * kTile * kTile);
  return fill >= (rounds > 1 ? 0.89 : k / kStageK <= 25 ? 0.55 : 0.72);
}

bool shapes_fit(int64_t rows, int64_t k, int64_t tokens) {
  return tokens > 0 && tokens <= (1 << 26) && rows > 0 && rows % 8 == 0 && rows <= (1 << 20) && k >= 4 * kStageK && k % kStageK == 0 && k <= (1 << 20) &&
         (rows + kTile - 1) / kTile * ((tokens + kTile - 1) / kTile) <= (1 << 30);
}

}  // namespace
}  // namespace tf24

extern "C" int tf24_linear16_suits(int64_t rows, int64_t k, int64_t tokens) {
  return tf24::shapes_fit(rows, k, tokens) && tf24::suits(rows, k, tokens, tf24::compute_units());
}

extern "C" int tf24_linear16(const void* w, int64_t ldw, int w_strided, const void* x, int64_t ldx, int dtype, int64_t rows, int64_t k, int64_t tokens,
                             void* y, int64_t ldy, const void* bias, void* stream) {
  using namespace tf24;
  const char* fn = "tf24_linear16";
  if (dtype != TF24_F16 && dtype != TF24_BF16) return fail(TF24_ERR_DTYPE, "%s: unsupported dtype %d", fn, dtype);
  if (!shapes_fit(rows, k, tokens))
    return fail(TF24_ERR_SHAPE, "%s: %lld rows x %lld against %lld tokens: rows must be a multiple of 8, k one of %d and at least %d", fn, (long long)rows, (long long)k,
                (long long)tokens, kStageK, 4 * kStageK);
  // a stage of a tile is addressed by 32-bit lane offsets
  if (ldw < (w_strided ? rows : k) || ldw % 8 || ldw > (1 << 22) || ldx < k || ldx % 8 || ldx > (1 << 22) || ldy < rows || ldy % 8)
    return fail(TF24_ERR_STRIDE, "%s: leading dimensions %lld, %lld, %lld must cover the rows, be multiples of 8 and at most %d", fn, (long long)ldw, (long long)ldx,
                (long long)ldy, 1 << 22);
  if (!w || !x || !y) return fail(TF24_ERR_ARG, "%s: null pointer", fn);
  if (int rc = check_aligned(fn, 16, {w, x, y})) return rc;
  if (int rc = check_aligned(fn, 2, {bias})) return rc;
  auto* go = dtype == TF24_F16 ? launch_linear<f16_t> : launch_linear<bf16_t>;
  return go(w, ldw, w_strided != 0, x, ldx, rows, k, tokens, y, ldy, bias, (hipStream_t)stream);
}
