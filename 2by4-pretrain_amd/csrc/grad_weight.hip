// Weight and bias gradient of a linear layer with a dense weight, 16-bit operands, float32 accumulation:
//
//     dW[i, j] = sum_t G[t, i] * X[t, j]        db[i] = sum_t G[t, i]
//
// G [tokens, m] and X [tokens, n] are read as they lie: the summed axis is the slow one of both.
//
// Bound by the matrix cores, and at this size by the power that they may draw: 12288 tokens, 3072 x 768 bf16 take 62
// us with db on one card (0.94 PFLOP/s; on 32 x 32 instructions 65, on 256 x 256 tiles 69, of zeros 55 on any; another card took 69.6 and
// 72.3 for the first two), where the library's product takes 110 to 140 us and its row sum 20 to 29.
//
// A block multiplies a 256(i) x 256(j) tile over a piece of the token axis: eight waves (2 along i x 4 along j), two per
// SIMD, wave tile 128 x 64 = 4 x 2 V_MFMA_F32_32X32X16.  (Four waves of 128 x 128 read a third less LDS, but nothing covers
// their waits: 0.53 instead of 0.50 us per stage, and 6 us more to fill and drain.)  Or a 192 x 192 tile on four waves (2 x 2,
// wave tile 96 x 96), which takes 0.36 us a stage: see choose_pieces.  32 tokens of both operands are one
// stage of 32 KB (24); five stages rotate through the LDS.  At the start of stage s the copies of s+1 and s+2 are in
// flight and those of s+3 go into the buffer of stage s-2, whose fragments every wave has used up before the barrier of
// stage s: no wave waits for its own reads there.
// Where takes_long says so, the 192 x 192 tiles take V_MFMA_F32_16X16X32 in stages of 64 tokens, three of which rotate: the copies of s+2 go
// into the buffer of stage s-1, so the barrier of stage s waits for the reads as well.
// Both operands need eight consecutive tokens of one column per lane: transposing reads (DS_READ_B64_TR_B16) of rows of
// 256 (192) columns.  16-byte chunks are XOR-swizzled by token so that the four tokens x 64 bytes that 32 lanes read touch every
// one of the 64 banks once (rows of 192 columns start half of the banks apart by themselves; with a swizzle that only spreads 16 lanes, half of the LDS cycles are conflicts).
// Few tiles and a long token axis: the axis is cut into pieces (choose_pieces); their float32 partial tiles are added in
// piece order by a second kernel, which rounds once.
#include "lds_copies.hpp"
#include <algorithm>
#include <type_traits>

namespace tf24 {
namespace {

typedef short short8v __attribute__((ext_vector_type(8)));

constexpr int kMaxPieces = 16;

// FR: rows and columns of the matrix instruction, 32 (16 tokens each) or 16 (32 tokens); a stage is two steps of that many tokens
template <int TILE_, int WAVES_J_, int FR_, int RING_>
struct TileT {
  static constexpr int TILE = TILE_, WAVES_J = WAVES_J_, WAVES = 2 * WAVES_J, THREADS = 64 * WAVES;
  static constexpr int FR = FR_, STEP_TOKENS = 512 / FR, STAGE_TOKENS = 2 * STEP_TOKENS, RING = RING_, AHEAD = RING == 5 ? 3 : 2;
  static constexpr int ROW_BYTES = TILE * 2, OPERAND = STAGE_TOKENS * ROW_BYTES, STAGE = 2 * OPERAND;
  static constexpr int CHUNKS = TILE / 8;                               // 16-byte chunks of a token's columns
  static constexpr int TI = TILE / 2 / FR, TJ = TILE / FR / WAVES_J;    // fragments of FR rows and of FR columns per wave
  static constexpr int SUMS = (TI + WAVES_J - 1) / WAVES_J;             // row fragments whose column sums a wave forms
  static constexpr int COPIES = OPERAND / 1024 / WAVES;                 // 1 KB copies per wave and operand of a stage
  static constexpr int MMA = TI * TJ, READS = 2 * (TI + TJ);                         // per step
  static constexpr int QUADS = FR * FR / 256, SLABS = QUADS * MMA;      // a lane's quads of four rows in a fragment and in all of a wave's
  static_assert(COPIES * 1024 * WAVES == OPERAND && MMA % COPIES == 0 && RING * STAGE <= 160 * 1024 && (RING == 5 || RING == 3), "a stage's copies divide among the waves");
  static __device__ __forceinline__ uint32_t swizzle(uint32_t token) {
    return TILE == 256 ? ((token & 3) << 2) | (((token >> 3) & 1) << 1) : (((token >> 1) & 1) << 2) | (((token >> 3) & 1) << 1);
  }
  // Rows of fragment ti of a wave: the waves that share rows hold their fragments rotated, so that the first SUMS of each are
  // (all but the last wave's, others: the same sums may be formed twice) another FR of them: those are the rows whose column
  // sums the wave forms.
  static __device__ __forceinline__ int fragment_row(int wave, int ti) {
    return (wave / WAVES_J) * (FR * TI) + ((ti + (wave % WAVES_J) * SUMS) % TI) * FR;
  }
  // where slab s of a wave's accumulators lies in the tile: four rows of one column per lane
  static __device__ __forceinline__ int slab_row(int wave, int lane, int s) {
    return fragment_row(wave, s / (QUADS * TJ)) + (s % QUADS) * 8 + (lane / FR) * 4;
  }
  static __device__ __forceinline__ int slab_col(int wave, int lane, int s) { return ((wave % WAVES_J) * TJ + (s / QUADS) % TJ) * FR + lane % FR; }
};
using Wide = TileT<256, 4, 32, 5>;
using Square = TileT<192, 2, 32, 5>;
using SquareLong = TileT<192, 2, 16, 3>;

__device__ __forceinline__ float16v mma(f16_t, short8v a, short8v b, float16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
}
__device__ __forceinline__ float16v mma(bf16_t, short8v a, short8v b, float16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ float4v mma(f16_t, short8v a, short8v b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
}
__device__ __forceinline__ float4v mma(bf16_t, short8v a, short8v b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ float widen(f16_t, short h) { return to_float(f16_t{(uint16_t)h}); }
__device__ __forceinline__ float widen(bf16_t, short h) { return to_float(bf16_t{(uint16_t)h}); }

// a sum rounded to the operands' type, as it is stored (float32 results hold the same values: a pass of its own that widens
// them, and one for db, are 5 us each)
template <typename T, typename OutT>
__device__ __forceinline__ OutT rounded(float v) {
  if constexpr (std::is_same<OutT, float>::value) return to_float(from_float<T>(v));
  else return from_float<T>(v);
}

struct Piece { int tile_i, tile_j, split; };
// units are (piece, tile), piece-major, the tiles of a piece column by column; see the kernel for the XCD order
__device__ __forceinline__ Piece locate(int unit, int tiles_i, int tiles_j) {
  const int ntiles = tiles_i * tiles_j, split = unit / ntiles, tile = unit - split * ntiles;
  return {tile / tiles_j, tile % tiles_j, split};
}

template <typename T, typename OutT, typename C, bool SUMS>
__global__ void __launch_bounds__(C::THREADS)
grad_weight_pipe(const uint8_t* __restrict__ g, int64_t ldg, const uint8_t* __restrict__ x, int64_t ldx, int64_t tokens,
                 int64_t m, int64_t n, int tiles_i, int tiles_j, int splits, float* __restrict__ partial, float* __restrict__ sums,
                 OutT* __restrict__ dw, OutT* __restrict__ db) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[C::RING * C::STAGE];
  // workgroup ids are dealt to the 8 XCDs round-robin: each XCD takes a run of units, which share operand columns in its L2
  const int nunits = tiles_i * tiles_j * splits, per_xcd = (nunits + 7) / 8;
  const int unit = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if (unit >= min(((int)(blockIdx.x & 7) + 1) * per_xcd, nunits)) return;
  const Piece at = locate(unit, tiles_i, tiles_j);
  const int64_t i0 = (int64_t)at.tile_i * C::TILE, j0 = (int64_t)at.tile_j * C::TILE;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wj = wave % C::WAVES_J;
  const int lrow = lane % C::FR, lblock = lane / C::FR;            // row or column of a fragment, block of eight tokens
  const int stages_all = (int)((tokens + C::STAGE_TOKENS - 1) / C::STAGE_TOKENS);
  const int st_begin = (int)((int64_t)at.split * stages_all / splits);
  const int nstages = (int)((int64_t)(at.split + 1) * stages_all / splits) - st_begin;
  // tokens of the last stage of the whole axis, if it is not a full one, and which stage of this piece that is (-1: none)
  const int ragged = (int)(tokens % C::STAGE_TOKENS);
  const int ragged_stage = ragged && st_begin + nstages == stages_all ? nstages - 1 : -1;

  // ---- copies: number q of a wave brings 1 KB of a stage (2 tokens of 256 columns); columns past the matrix re-read its last chunk
  const uint8_t* g_at = g + (int64_t)st_begin * C::STAGE_TOKENS * ldg;
  const uint8_t* x_at = x + (int64_t)st_begin * C::STAGE_TOKENS * ldx;
  const int64_t g_step = (int64_t)C::STAGE_TOKENS * ldg, x_step = (int64_t)C::STAGE_TOKENS * ldx;
  auto offset_of = [&](int q, int64_t c0, int64_t cols, int64_t ld, int rows) {
    const uint32_t chunk = (uint32_t)((wave * C::COPIES + q) * 64 + lane), token = chunk / C::CHUNKS;
    const int64_t col = min(c0 + (int64_t)((chunk % C::CHUNKS) ^ C::swizzle(token)) * 8, cols - 8);
    return (uint32_t)(min((int64_t)token, (int64_t)rows - 1) * ld + col * 2);
  };
  uint32_t og[C::COPIES], ox[C::COPIES];
#pragma unroll
  for (int q = 0; q < C::COPIES; q++) {
    og[q] = offset_of(q, i0, m, ldg, C::STAGE_TOKENS);
    ox[q] = offset_of(q, j0, n, ldx, C::STAGE_TOKENS);
  }
  const uint32_t smem_at = lds_offset(smem);
  auto copy_one = [&](int q, int st, uint32_t buf) {             // q: the wave's copies of G, then those of X
    const uint32_t dst = smem_at + buf + (uint32_t)(wave * C::COPIES + (q % C::COPIES)) * 1024;
    if (q < C::COPIES) g2l16(g_at + (int64_t)st * g_step, og[q], dst);
    else g2l16(x_at + (int64_t)st * x_step, ox[q - C::COPIES], dst + C::OPERAND);
  };
  auto copy_ragged = [&](int st, uint32_t buf) {                 // tokens past the last one re-read it (and are zeroed on arrival)
#pragma unroll
    for (int q = 0; q < C::COPIES; q++) {
      const uint32_t dst = smem_at + buf + (uint32_t)(wave * C::COPIES + q) * 1024;
      g2l16(g_at + (int64_t)st * g_step, offset_of(q, i0, m, ldg, ragged), dst);
      g2l16(x_at + (int64_t)st * x_step, offset_of(q, j0, n, ldx, ragged), dst + C::OPERAND);
    }
  };
  auto copy_stage = [&](int st, uint32_t buf) {
    if (st == ragged_stage) copy_ragged(st, buf);
    else {
#pragma unroll
      for (int q = 0; q < 2 * C::COPIES; q++) copy_one(q, st, buf);
    }
  };
  // stage st has arrived when this wave's copies of the (at most AHEAD - 1) stages behind it are all that is in flight; with three
  // buffers the next copies go into the stage just read, so the wave's reads of it are waited for as well
  constexpr bool READS_TOO = C::RING == 3;
  auto arrive = [&](int st, uint32_t buf) {
    const int behind = min(nstages - 1 - st, C::AHEAD - 1);
    if (behind >= 2) wait_copies_and_barrier<4 * C::COPIES, READS_TOO>();
    else if (behind == 1) wait_copies_and_barrier<2 * C::COPIES, READS_TOO>();
    else wait_copies_and_barrier<0, READS_TOO>();
    if (st == ragged_stage) {
      for (int c = tid; c < (C::STAGE_TOKENS - ragged) * (C::ROW_BYTES / 16); c += C::THREADS) {
        *reinterpret_cast<int4v*>(smem + buf + ragged * C::ROW_BYTES + c * 16) = int4v{0, 0, 0, 0};
        *reinterpret_cast<int4v*>(smem + buf + C::OPERAND + ragged * C::ROW_BYTES + c * 16) = int4v{0, 0, 0, 0};
      }
      __syncthreads();
    }
  };

  std::conditional_t<C::FR == 32, float16v, float4v> acc[C::TI][C::TJ];
#pragma unroll
  for (int ti = 0; ti < C::TI; ti++)
#pragma unroll
    for (int tj = 0; tj < C::TJ; tj++)
#pragma unroll
      for (int r = 0; r < 4 * C::QUADS; r++) acc[ti][tj][r] = 0.0f;

  // ---- fragments: in a group of 16 lanes, lane i receives the halfwords i % 4 of the source lanes 4e + i / 4 (e = 0..3).
  // Source lane s addresses token t0 + s / 4, columns 4 * (s % 4).. of the group's 16, so lane i gets tokens t0..t0+3 of
  // column i; the lanes of block b of FR lanes take tokens 8b .. 8b + 7 of an instruction's (t0 = 8b, 8b + 4).
  const int s16 = lane & 15, jbase = C::FR == 32 ? ((lane >> 4) & 1) * 16 : 0;
  const uint32_t token0 = (uint32_t)(lblock * 8 + (s16 >> 2));
  uint32_t a_off[C::TI], b_off[C::TJ];
#pragma unroll
  for (int f = 0; f < C::TI; f++) {
    const uint32_t c = (uint32_t)(C::fragment_row(wave, f) + jbase + (s16 & 3) * 4);
    a_off[f] = token0 * C::ROW_BYTES + (((c >> 3) ^ C::swizzle(token0)) * 16) + ((c >> 2) & 1) * 8;
  }
#pragma unroll
  for (int f = 0; f < C::TJ; f++) {
    const uint32_t c = (uint32_t)((wj * C::TJ + f) * C::FR + jbase + (s16 & 3) * 4);
    b_off[f] = C::OPERAND + token0 * C::ROW_BYTES + (((c >> 3) ^ C::swizzle(token0)) * 16) + ((c >> 2) & 1) * 8;
  }
  // the reads of a step in the order in which the next step's instructions need them: G's fragment 0, X's, G's others
  short4v af[2][C::TI][2], bf[2][C::TJ][2];
  auto read_one = [&](int set, int q, uint32_t buf, int step) {
    const uint8_t* base = smem + buf + step * (C::STEP_TOKENS * C::ROW_BYTES) + (q & 1) * (4 * C::ROW_BYTES);
    const int f = q >> 1;
    if (f >= 1 && f <= C::TJ) bf[set][f - 1][q & 1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(lds_ptr_t)(base + b_off[f - 1]));
    else af[set][f ? f - C::TJ : 0][q & 1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(lds_ptr_t)(base + a_off[f ? f - C::TJ : 0]));
  };
  // Column sums of G: one element (of 192 x 192 tiles two) behind each matrix instruction (two vector instructions under 32 cycles of it), by the
  // blocks of every tile column: a branch here would make the compiler wait for all reads in flight.
  float colsum[C::SUMS] = {};
  constexpr int PER_MMA = (8 * C::SUMS + C::MMA - 1) / C::MMA;
  // The instructions of a step from one register set; behind each of them one read of the next step into the other set
  // and, over the two steps of a stage, the copies of stage cst.
  auto mma_step = [&](int set, bool reads, uint32_t src, int rstep, int half, bool copies, int cst, uint32_t dst) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < C::MMA; i++) {
      const int ti = i / C::TJ, tj = i % C::TJ;
      const short8v a = __builtin_shufflevector(af[set][ti][0], af[set][ti][1], 0, 1, 2, 3, 4, 5, 6, 7);
      const short8v b = __builtin_shufflevector(bf[set][tj][0], bf[set][tj][1], 0, 1, 2, 3, 4, 5, 6, 7);
      acc[ti][tj] = mma(T{}, a, b, acc[ti][tj]);
      __builtin_amdgcn_sched_barrier(0);
      if (reads) {
#pragma unroll
        for (int q = i * C::READS / C::MMA; q < (i + 1) * C::READS / C::MMA; q++) read_one(set ^ 1, q, src, rstep);
      }
      if (copies && (i + 1) % (C::MMA / C::COPIES) == 0) copy_one(half * C::COPIES + i / (C::MMA / C::COPIES), cst, dst);
      if constexpr (SUMS) {
#pragma unroll
        for (int e = i * PER_MMA; e < (i + 1) * PER_MMA && e < 8 * C::SUMS; e++) {
          colsum[e >> 3] += widen(T{}, af[set][e >> 3][(e >> 2) & 1][e & 3]);
          asm volatile("" : "+v"(colsum[e >> 3]));               // (kept here: moved together they would run after the last instruction)
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto next_buf = [](uint32_t b) { return b + C::STAGE == C::RING * C::STAGE ? 0u : b + C::STAGE; };

  copy_stage(0, 0);
  if (nstages > 1) copy_stage(1, C::STAGE);
  if (C::AHEAD > 2 && nstages > 2) copy_stage(2, 2 * C::STAGE);
  arrive(0, 0);
#pragma unroll
  for (int q = 0; q < C::READS; q++) read_one(0, q, 0, 0);
  uint32_t cur = 0, far = C::AHEAD * C::STAGE;                     // buffers of stage st and of stage st + AHEAD
  if (nstages > C::AHEAD) copy_stage(C::AHEAD, far);
  mma_step(0, true, cur, 1, 0, false, 0, 0);
  const int whole = ragged_stage < 0 ? nstages : nstages - 1;    // stages whose copies take the common form
  int st = 1;
  for (; st + C::AHEAD < whole; st++) {
    cur = next_buf(cur); far = next_buf(far);
    wait_copies_and_barrier<(C::AHEAD - 1) * 2 * C::COPIES, READS_TOO>();
    mma_step(1, true, cur, 0, 0, true, st + C::AHEAD, far);      // the last step of stage st - 1
    mma_step(0, true, cur, 1, 1, true, st + C::AHEAD, far);
  }
  for (; st < nstages; st++) {
    cur = next_buf(cur); far = next_buf(far);
    arrive(st, cur);
    if (st + C::AHEAD < nstages) copy_ragged(st + C::AHEAD, far);
    mma_step(1, true, cur, 0, 0, false, 0, 0);
    mma_step(0, true, cur, 1, 0, false, 0, 0);
  }
  mma_step(1, false, 0, 0, 0, false, 0, 0);

  if (SUMS && at.tile_j == 0) {
#pragma unroll
    for (int h = 0; h < C::SUMS; h++) {
      float v = colsum[h];
      if (C::FR == 16) v += __shfl_xor(v, 16);
      v += __shfl_xor(v, 32);
      const int64_t row = i0 + C::fragment_row(wave, h) + lrow;
      if (lblock == 0) {
        if (splits > 1) sums[(int64_t)at.split * tiles_i * C::TILE + row] = v;
        else if (row < m) db[row] = rounded<T, OutT>(v);
      }
    }
  }
  if (splits > 1) {                                              // slab (fragment, quarter) of the tile: 4 rows of one column per lane
    float* out = partial + (int64_t)unit * (C::TILE * C::TILE) + tid * 4;
#pragma unroll
    for (int s = 0; s < C::SLABS; s++) {
      const auto& v = acc[s / (C::QUADS * C::TJ)][s / C::QUADS % C::TJ];
      const int r = s % C::QUADS * 4;
      *reinterpret_cast<float4v*>(out + s * (C::THREADS * 4)) = float4v{v[r], v[r + 1], v[r + 2], v[r + 3]};
    }
    return;
  }
#pragma unroll
  for (int s = 0; s < C::SLABS; s++) {
    const int64_t row = i0 + C::slab_row(wave, lane, s), col = j0 + C::slab_col(wave, lane, s);
    if (row < m && col < n) {
#pragma unroll
      for (int r = 0; r < 4; r++) dw[(row + r) * n + col] = rounded<T, OutT>(acc[s / (C::QUADS * C::TJ)][s / C::QUADS % C::TJ][s % C::QUADS * 4 + r]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// dW and db from the pieces: block (tile, slab), and with blockIdx.x one past the tiles the sums of the columns
template <typename T, typename OutT, typename C>
__global__ void __launch_bounds__(C::THREADS)
grad_weight_reduce(const float* __restrict__ partial, const float* __restrict__ sums, int splits, int64_t m, int64_t n, int tiles_i, int tiles_j,
                   OutT* __restrict__ dw, OutT* __restrict__ db) {
  const int ntiles = tiles_i * tiles_j, tid = threadIdx.x;
  if ((int)blockIdx.x == ntiles) {
    for (int64_t i = (int64_t)blockIdx.y * C::THREADS + tid; i < m; i += (int64_t)gridDim.y * C::THREADS) {
      float v = 0.0f;
      for (int p = 0; p < splits; p++) v += sums[(int64_t)p * tiles_i * C::TILE + i];
      db[i] = rounded<T, OutT>(v);
    }
    return;
  }
  const Piece at = locate((int)blockIdx.x, tiles_i, tiles_j);
  const int lane = tid & 63, wave = tid >> 6, s = (int)blockIdx.y;
  const int64_t row = (int64_t)at.tile_i * C::TILE + C::slab_row(wave, lane, s), col = (int64_t)at.tile_j * C::TILE + C::slab_col(wave, lane, s);
  if (row >= m || col >= n) return;
  const float* first = partial + (int64_t)blockIdx.x * (C::TILE * C::TILE) + s * (C::THREADS * 4) + tid * 4;
  const int64_t piece = (int64_t)ntiles * (C::TILE * C::TILE);
  float4v v = {0, 0, 0, 0};
  for (int p0 = 0; p0 < splits; p0 += 8) {                       // eight independent loads in flight
    float4v part[8];
#pragma unroll
    for (int u = 0; u < 8; u++) part[u] = *reinterpret_cast<const float4v*>(first + (int64_t)min(p0 + u, splits - 1) * piece);
#pragma unroll
    for (int u = 0; u < 8; u++)
      if (p0 + u < splits) v += part[u];
  }
#pragma unroll
  for (int r = 0; r < 4; r++) dw[(row + r) * n + col] = rounded<T, OutT>(v[r]);
}

template <typename C>
int64_t piece_bytes(int64_t tiles_i, int64_t tiles_j) { return (tiles_i * tiles_j * C::TILE + tiles_i) * C::TILE * 4; }

// The number of pieces with the least  stages of one piece x STAGE_US + (more than one: 3 us + 0.32 us per MB of partial tiles),
// all in one round of the compute units.  The constants are fitted to timings of 1 to 16 pieces over 500 to 16384 tokens
// and 2048 x 512 to 6400 x 1600 outputs; the choice is within 4 % of the best on all of them.  More than 128 tiles stay in one
// piece, since two would need a second round of the compute units (against the library's product see _linear16).  3072 x 768, us:
// 12288 tokens, 36 tiles of 256 x 256, 209 in one piece, 82 in three, 70 in seven; 64 tiles of 192 x 192, 96 in two, 73 in three,
// 67 in four; 1024 tokens 24 in one piece of the wide tiles and 30 in seven.
// 192 x 192 tiles where the same estimate is the lesser with them (takes_square): as many compute units with fewer pieces, and
// the partial sums are what the pieces cost.  Of 30 outputs of 500 to 12288 tokens they are the faster ones for 23, by 9 % over
// all: 3072 x 768 over 745 tokens 18.9 -> 15.7 us, over 2916 31.4 -> 27.5, over 12288 70.2 -> 67; 6400 x 1600 over 2781, 306
// of them instead of 175, would take 88 for 63.
struct Pieces { int count; double us; };
template <typename C>
Pieces choose_pieces(int64_t tokens, int64_t m, int64_t n, int64_t workspace_bytes) {
  constexpr double STAGE_US = std::is_same<C, Wide>::value ? 0.6 : 0.36;               // of 32 tokens
  const int64_t tiles_i = (m + C::TILE - 1) / C::TILE, tiles_j = (n + C::TILE - 1) / C::TILE;
  const int64_t stages = (tokens + 31) / 32, tiles = tiles_i * tiles_j;
  Pieces best{1, (double)(stages * ((tiles + 255) / 256)) * STAGE_US};
  for (int64_t p = 2; p <= kMaxPieces && p <= stages / 4 && p * tiles <= 256 && p * piece_bytes<C>(tiles_i, tiles_j) <= workspace_bytes; p++) {
    const double us = (double)((stages + p - 1) / p) * STAGE_US + 3.0 + (double)(p * tiles) * (C::TILE * C::TILE * 4e-6 * 0.32);
    if (us < best.us) best = {(int)p, us};
  }
  return best;
}
bool takes_square(int64_t tokens, int64_t m, int64_t n, int64_t workspace_bytes) {
  return choose_pieces<Square>(tokens, m, n, workspace_bytes).us < 0.97 * choose_pieces<Wide>(tokens, m, n, workspace_bytes).us;
}

// 192 x 192 tiles of at least kLongTokens tokens on at least kLongBlocks compute units are bound by power, and take 16 x 16 instructions: alone, on
// random operands in registers, those sustain 1.9 PFLOP/s where the 32 x 32 ones do 1.65.  Their stages are of 64 tokens, three buffers of
// 48 KB.  us on 32 x 32 instructions and on these: 3072 x 768 over 12288 tokens (256 blocks of 3072) 65.2 and 62.5, 768 x 3072 65.5 and 63.7,
// 2048 x 512 over 16384 (231 of 2340) 48.9 and 47.5, 5120 x 1280 over 4423 (189 of 4423) 65.8 and 63.9; fewer blocks or tokens, where the longer
// first stage shows: 1024 x 4096 over 2000 (132 of 2000) 32.8 and 33.7, 3072 x 768 over 745 16.9 and 17.4, 512 x 2048 over 5000 24.6 and 25.2.
constexpr int64_t kLongTokens = 1024, kLongBlocks = 160;
bool takes_long(int64_t tokens, int64_t m, int64_t n, int64_t workspace_bytes) {
  const int64_t pieces = choose_pieces<Square>(tokens, m, n, workspace_bytes).count;
  const int64_t tiles = (m + Square::TILE - 1) / Square::TILE * ((n + Square::TILE - 1) / Square::TILE);
  return tiles * pieces >= kLongBlocks && tokens >= kLongTokens * pieces;
}

template <typename T, typename OutT, typename C>
int launch(const void* g, int64_t ldg, const void* x, int64_t ldx, int64_t tokens, int64_t m, int64_t n, void* dw, void* db,
           void* workspace, int64_t workspace_bytes, hipStream_t s) {
  const int tiles_i = (int)((m + C::TILE - 1) / C::TILE), tiles_j = (int)((n + C::TILE - 1) / C::TILE);
  const int pieces = workspace ? choose_pieces<C>(tokens, m, n, workspace_bytes).count : 1;
  float* partial = (float*)workspace;
  float* sums = pieces > 1 ? partial + (int64_t)pieces * tiles_i * tiles_j * C::TILE * C::TILE : nullptr;     // behind the partial tiles
  const int per_xcd = (tiles_i * tiles_j * pieces + 7) / 8;
  auto pipe = [&](auto with_sums) {
    hipLaunchKernelGGL((grad_weight_pipe<T, OutT, C, decltype(with_sums)::value>), dim3((unsigned)(per_xcd * 8)), dim3(C::THREADS), 0, s, (const uint8_t*)g, ldg * 2,
                       (const uint8_t*)x, ldx * 2, tokens, m, n, tiles_i, tiles_j, pieces, partial, sums, (OutT*)dw, (OutT*)db);
  };
  if (db) pipe(std::true_type{}); else pipe(std::false_type{});
  if (pieces > 1)
    hipLaunchKernelGGL((grad_weight_reduce<T, OutT, C>), dim3((unsigned)(tiles_i * tiles_j + (db ? 1 : 0)), C::SLABS), dim3(C::THREADS), 0, s, partial, sums, pieces, m, n,
                       tiles_i, tiles_j, (OutT*)dw, (OutT*)db);
  return check_launch("tf24_grad_weight");
}

template <typename T, typename OutT>
int launch_either(const void* g, int64_t ldg, const void* x, int64_t ldx, int64_t tokens, int64_t m, int64_t n, void* dw, void* db,
                  void* workspace, int64_t workspace_bytes, hipStream_t s) {
  const int64_t bytes = workspace ? workspace_bytes : 0;
  auto* go = !takes_square(tokens, m, n, bytes) ? launch<T, OutT, Wide> : takes_long(tokens, m, n, bytes) ? launch<T, OutT, SquareLong> : launch<T, OutT, Square>;
  return go(g, ldg, x, ldx, tokens, m, n, dw, db, workspace, workspace_bytes, s);
}

template <typename C>
int64_t bytes_wanted(int64_t tokens, int64_t m, int64_t n) {
  const int pieces = choose_pieces<C>(tokens, m, n, (int64_t)1 << 40).count;
  return pieces > 1 ? pieces * piece_bytes<C>((m + C::TILE - 1) / C::TILE, (n + C::TILE - 1) / C::TILE) : 0;
}

}  // namespace
}  // namespace tf24

extern "C" int64_t tf24_grad_weight_workspace_bytes(int64_t tokens, int64_t m, int64_t n) {
  using namespace tf24;
  if (tokens <= 0 || m <= 0 || n <= 0) return 0;
  return takes_square(tokens, m, n, (int64_t)1 << 40) ? bytes_wanted<Square>(tokens, m, n) : bytes_wanted<Wide>(tokens, m, n);
}

namespace tf24 {
namespace {
int run(const char* fn, bool f32, const void* g, int64_t ldg, const void* x, int64_t ldx, int dtype, int64_t tokens, int64_t m, int64_t n,
        void* dw, void* db, void* workspace, int64_t workspace_bytes, void* stream) {
  if (dtype != TF24_F16 && dtype != TF24_BF16) return fail(TF24_ERR_DTYPE, "%s: unsupported dtype %d", fn, dtype);
  if (tokens <= 0 || tokens > 0x7fffffffLL) return fail(TF24_ERR_SHAPE, "%s: bad number of tokens %lld", fn, (long long)tokens);
  if (m <= 0 || m % 8 || n <= 0 || n % 8 || m > (1 << 20) || n > (1 << 20))
    return fail(TF24_ERR_SHAPE, "%s: %lld x %lld must be positive multiples of 8, at most %d", fn, (long long)m, (long long)n, 1 << 20);
  // a stage's tokens, 32 or 64, are addressed by 32-bit lane offsets
  if (ldg < m || ldg % 8 || ldg > (1 << 23) || ldx < n || ldx % 8 || ldx > (1 << 23))
    return fail(TF24_ERR_STRIDE, "%s: leading dimensions %lld, %lld must cover the rows, be multiples of 8 and at most %d", fn, (long long)ldg, (long long)ldx, 1 << 23);
  if (!g || !x || !dw) return fail(TF24_ERR_ARG, "%s: null pointer", fn);
  if (workspace_bytes < 0) return fail(TF24_ERR_ARG, "%s: negative workspace size", fn);
  if (int rc = check_aligned(fn, 16, {g, x, workspace})) return rc;
  if (int rc = check_aligned(fn, f32 ? 4 : 2, {dw, db})) return rc;
  hipStream_t s = (hipStream_t)stream;
  auto* go = dtype == TF24_F16 ? (f32 ? launch_either<f16_t, float> : launch_either<f16_t, f16_t>)
                               : (f32 ? launch_either<bf16_t, float> : launch_either<bf16_t, bf16_t>);
  return go(g, ldg, x, ldx, tokens, m, n, dw, db, workspace, workspace_bytes, s);
}
}  // namespace
}  // namespace tf24

extern "C" int tf24_grad_weight(const void* g, int64_t ldg, const void* x, int64_t ldx, int dtype, int64_t tokens, int64_t m, int64_t n,
                                void* dw, void* db, void* workspace, int64_t workspace_bytes, void* stream) {
  return tf24::run("tf24_grad_weight", false, g, ldg, x, ldx, dtype, tokens, m, n, dw, db, workspace, workspace_bytes, stream);
}

extern "C" int tf24_grad_weight_f32(const void* g, int64_t ldg, const void* x, int64_t ldx, int dtype, int64_t tokens, int64_t m, int64_t n,
                                    float* dw, float* db, void* workspace, int64_t workspace_bytes, void* stream) {
  return tf24::run("tf24_grad_weight_f32", true, g, ldg, x, ldx, dtype, tokens, m, n, dw, db, workspace, workspace_bytes, stream);
}
