// Weight and bias gradient of a linear layer with a dense weight, 16-bit operands, float32 accumulation:
//
//     dW[i, j] = sum_t G[t, i] * X[t, j]        db[i] = sum_t G[t, i]
//
// G [tokens, m] and X [tokens, n] are read as they lie: the summed axis is the slow one of both.
//
// Bound by the matrix cores, and at this size by the power that they may draw: 12288 tokens, 3072 x 768 bf16 take 67 to
// 72 us with db (0.8 PFLOP/s; 54 us on matrices of zeros), where the library's product takes 125 to 140 us and its row sum 29.
//
// A block multiplies a 256(i) x 256(j) tile over a piece of the token axis: eight waves (2 along i x 4 along j), two per
// SIMD, wave tile 128 x 64 = 4 x 2 V_MFMA_F32_32X32X16.  (Four waves of 128 x 128 read a third less LDS, but nothing covers
// their waits: 0.53 instead of 0.50 us per stage, and 6 us more to fill and drain.)  32 tokens of both operands are one
// stage of 32 KB; five stages rotate through the 160 KB of LDS.  At the start of stage s the copies of s+1 and s+2 are in
// flight and those of s+3 go into the buffer of stage s-2, whose fragments every wave has used up before the barrier of
// stage s: no wave waits for its own reads there.
// Both operands need eight consecutive tokens of one column per lane: transposing reads (DS_READ_B64_TR_B16) of rows of
// 256 columns.  16-byte chunks are XOR-swizzled by token so that the four tokens x 64 bytes that 32 lanes read touch every
// one of the 64 banks once (with a swizzle that only spreads 16 lanes, half of the LDS cycles are conflicts).
// Few tiles and a long token axis: the axis is cut into pieces (choose_pieces); their float32 partial tiles are added in
// piece order by a second kernel, which rounds once.
#include "lds_copies.hpp"
#include <algorithm>
#include <type_traits>

namespace tf24 {
namespace {

typedef short short8v __attribute__((ext_vector_type(8)));

constexpr int kTile = 256, kStageTokens = 32, kRing = 5;
constexpr int kRowBytes = kTile * 2, kOperand = kStageTokens * kRowBytes, kStage = 2 * kOperand;
constexpr int kWavesJ = 4, kThreads = 128 * kWavesJ;
constexpr int kTJ = 8 / kWavesJ;                                        // fragments of 32 columns per wave (and 4 of 32 rows)
constexpr int kSums = 4 / kWavesJ;                                      // row fragments whose column sums a wave forms
constexpr int kCopies = kOperand / 1024 / (2 * kWavesJ);                // 1 KB copies per wave and operand of a stage
constexpr int kMma = 4 * kTJ, kReads = 2 * (4 + kTJ), kSlabs = 4 * kMma; // per step of 16 tokens; quarters of a wave's fragments
constexpr int kMaxPieces = 16;

__device__ __forceinline__ float16v mma(f16_t, short8v a, short8v b, float16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
}
__device__ __forceinline__ float16v mma(bf16_t, short8v a, short8v b, float16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ float widen(f16_t, short h) { return to_float(f16_t{(uint16_t)h}); }
__device__ __forceinline__ float widen(bf16_t, short h) { return to_float(bf16_t{(uint16_t)h}); }

__device__ __forceinline__ uint32_t swizzle(uint32_t token) { return ((token & 3) << 2) | (((token >> 3) & 1) << 1); }

// Rows of fragment ti of a wave: the four waves that share 128 rows hold their fragments rotated, so that fragment 0 of
// each is another 32 of them: those are the rows whose column sums the wave forms.
__device__ __forceinline__ int fragment_row(int wave, int ti) { return (wave / kWavesJ) * 128 + ((ti + (wave % kWavesJ) * kSums) & 3) * 32; }

struct Piece { int tile_i, tile_j, split; };
// units are (piece, tile), piece-major, the tiles of a piece column by column; see the kernel for the XCD order
__device__ __forceinline__ Piece locate(int unit, int tiles_i, int tiles_j) {
  const int ntiles = tiles_i * tiles_j, split = unit / ntiles, tile = unit - split * ntiles;
  return {tile / tiles_j, tile % tiles_j, split};
}

template <typename T, bool SUMS>
__global__ void __launch_bounds__(kThreads)
grad_weight_pipe(const uint8_t* __restrict__ g, int64_t ldg, const uint8_t* __restrict__ x, int64_t ldx, int64_t tokens,
                 int64_t m, int64_t n, int tiles_i, int tiles_j, int splits, float* __restrict__ partial, float* __restrict__ sums,
                 T* __restrict__ dw, T* __restrict__ db) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kRing * kStage];
  // workgroup ids are dealt to the 8 XCDs round-robin: each XCD takes a run of units, which share operand columns in its L2
  const int nunits = tiles_i * tiles_j * splits, per_xcd = (nunits + 7) / 8;
  const int unit = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if (unit >= min(((int)(blockIdx.x & 7) + 1) * per_xcd, nunits)) return;
  const Piece at = locate(unit, tiles_i, tiles_j);
  const int64_t i0 = (int64_t)at.tile_i * kTile, j0 = (int64_t)at.tile_j * kTile;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wj = wave % kWavesJ;
  const int l32 = lane & 31, lh = lane >> 5;
  const int stages_all = (int)((tokens + kStageTokens - 1) / kStageTokens);
  const int st_begin = (int)((int64_t)at.split * stages_all / splits);
  const int nstages = (int)((int64_t)(at.split + 1) * stages_all / splits) - st_begin;
  // tokens of the last stage of the whole axis, if it is not a full one, and which stage of this piece that is (-1: none)
  const int ragged = (int)(tokens % kStageTokens);
  const int ragged_stage = ragged && st_begin + nstages == stages_all ? nstages - 1 : -1;

  // ---- copies: number q of a wave brings 2 tokens x 512 bytes; columns past the matrix re-read its last chunk
  const uint8_t* g_at = g + (int64_t)st_begin * kStageTokens * ldg;
  const uint8_t* x_at = x + (int64_t)st_begin * kStageTokens * ldx;
  const int64_t g_step = (int64_t)kStageTokens * ldg, x_step = (int64_t)kStageTokens * ldx;
  auto offset_of = [&](int q, int64_t c0, int64_t cols, int64_t ld, int rows) {
    const uint32_t token = (uint32_t)((wave * kCopies + q) * 2 + lh);
    const int64_t col = min(c0 + (int64_t)((uint32_t)l32 ^ swizzle(token)) * 8, cols - 8);
    return (uint32_t)(min((int64_t)token, (int64_t)rows - 1) * ld + col * 2);
  };
  uint32_t og[kCopies], ox[kCopies];
#pragma unroll
  for (int q = 0; q < kCopies; q++) {
    og[q] = offset_of(q, i0, m, ldg, kStageTokens);
    ox[q] = offset_of(q, j0, n, ldx, kStageTokens);
  }
  const uint32_t smem_at = lds_offset(smem);
  auto copy_one = [&](int q, int st, uint32_t buf) {             // q: the wave's copies of G, then those of X
    const uint32_t dst = smem_at + buf + (uint32_t)(wave * kCopies + (q % kCopies)) * 1024;
    if (q < kCopies) g2l16(g_at + (int64_t)st * g_step, og[q], dst);
    else g2l16(x_at + (int64_t)st * x_step, ox[q - kCopies], dst + kOperand);
  };
  auto copy_ragged = [&](int st, uint32_t buf) {                 // tokens past the last one re-read it (and are zeroed on arrival)
#pragma unroll
    for (int q = 0; q < kCopies; q++) {
      const uint32_t dst = smem_at + buf + (uint32_t)(wave * kCopies + q) * 1024;
      g2l16(g_at + (int64_t)st * g_step, offset_of(q, i0, m, ldg, ragged), dst);
      g2l16(x_at + (int64_t)st * x_step, offset_of(q, j0, n, ldx, ragged), dst + kOperand);
    }
  };
  auto copy_stage = [&](int st, uint32_t buf) {
    if (st == ragged_stage) copy_ragged(st, buf);
    else {
#pragma unroll
      for (int q = 0; q < 2 * kCopies; q++) copy_one(q, st, buf);
    }
  };
  // stage st has arrived when this wave's copies of the (at most two) stages behind it are all that is in flight
  auto arrive = [&](int st, uint32_t buf) {
    const int behind = nstages - 1 - st;
    if (behind >= 2) wait_copies_and_barrier<4 * kCopies, false>();
    else if (behind == 1) wait_copies_and_barrier<2 * kCopies, false>();
    else wait_copies_and_barrier<0, false>();
    if (st == ragged_stage) {
      for (int c = tid; c < (kStageTokens - ragged) * (kRowBytes / 16); c += kThreads) {
        *reinterpret_cast<int4v*>(smem + buf + ragged * kRowBytes + c * 16) = int4v{0, 0, 0, 0};
        *reinterpret_cast<int4v*>(smem + buf + kOperand + ragged * kRowBytes + c * 16) = int4v{0, 0, 0, 0};
      }
      __syncthreads();
    }
  };

  float16v acc[4][kTJ];
#pragma unroll
  for (int ti = 0; ti < 4; ti++)
#pragma unroll
    for (int tj = 0; tj < kTJ; tj++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[ti][tj][r] = 0.0f;

  // ---- fragments: in a group of 16 lanes, lane i receives the halfwords i % 4 of the source lanes 4e + i / 4 (e = 0..3).
  // Source lane s addresses token t0 + s / 4, columns 4 * (s % 4).. of the group's 16, so lane i gets tokens t0..t0+3 of
  // column i; lanes 0..31 take tokens 0..7 of an instruction's 16 (t0 = 0, 4), lanes 32..63 tokens 8..15.
  const int s16 = lane & 15, jbase = ((lane >> 4) & 1) * 16;
  const uint32_t token0 = (uint32_t)(lh * 8 + (s16 >> 2));
  uint32_t a_off[4], b_off[kTJ];
#pragma unroll
  for (int f = 0; f < 4; f++) {
    const uint32_t c = (uint32_t)(fragment_row(wave, f) + jbase + (s16 & 3) * 4);
    a_off[f] = token0 * kRowBytes + (((c >> 3) ^ swizzle(token0)) * 16) + ((c >> 2) & 1) * 8;
  }
#pragma unroll
  for (int f = 0; f < kTJ; f++) {
    const uint32_t c = (uint32_t)((wj * kTJ + f) * 32 + jbase + (s16 & 3) * 4);
    b_off[f] = kOperand + token0 * kRowBytes + (((c >> 3) ^ swizzle(token0)) * 16) + ((c >> 2) & 1) * 8;
  }
  // the reads of a step in the order in which the next step's instructions need them: G's fragment 0, X's, G's others
  short4v af[2][4][2], bf[2][kTJ][2];
  auto read_one = [&](int set, int q, uint32_t buf, int step) {
    const uint8_t* base = smem + buf + step * (16 * kRowBytes) + (q & 1) * (4 * kRowBytes);
    const int f = q >> 1;
    if (f >= 1 && f <= kTJ) bf[set][f - 1][q & 1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(lds_ptr_t)(base + b_off[f - 1]));
    else af[set][f ? f - kTJ : 0][q & 1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(lds_ptr_t)(base + a_off[f ? f - kTJ : 0]));
  };
  // Column sums of G: one element behind each matrix instruction (two vector instructions under 32 cycles of it), by the
  // blocks of every tile column: a branch here would make the compiler wait for all reads in flight.
  float colsum[kSums] = {};
  // The instructions of a step from one register set; behind each of them one read of the next step into the other set
  // and, over the two steps of a stage, the copies of stage cst.
  auto mma_step = [&](int set, bool reads, uint32_t src, int rstep, int half, bool copies, int cst, uint32_t dst) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kMma; i++) {
      const int ti = i / kTJ, tj = i % kTJ;
      const short8v a = __builtin_shufflevector(af[set][ti][0], af[set][ti][1], 0, 1, 2, 3, 4, 5, 6, 7);
      const short8v b = __builtin_shufflevector(bf[set][tj][0], bf[set][tj][1], 0, 1, 2, 3, 4, 5, 6, 7);
      acc[ti][tj] = mma(T{}, a, b, acc[ti][tj]);
      __builtin_amdgcn_sched_barrier(0);
      if (reads) {
#pragma unroll
        for (int q = i * kReads / kMma; q < (i + 1) * kReads / kMma; q++) read_one(set ^ 1, q, src, rstep);
      }
      if (copies && (i + 1) % (kMma / kCopies) == 0) copy_one(half * kCopies + i / (kMma / kCopies), cst, dst);
      if constexpr (SUMS) {
        colsum[i >> 3] += widen(T{}, af[set][i >> 3][(i >> 2) & 1][i & 3]);
        asm volatile("" : "+v"(colsum[i >> 3]));                 // (kept here: moved together they would run after the last instruction)
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto next_buf = [](uint32_t b) { return b + kStage == kRing * kStage ? 0u : b + kStage; };

  copy_stage(0, 0);
  if (nstages > 1) copy_stage(1, kStage);
  if (nstages > 2) copy_stage(2, 2 * kStage);
  arrive(0, 0);
#pragma unroll
  for (int q = 0; q < kReads; q++) read_one(0, q, 0, 0);
  uint32_t cur = 0, far = 3 * kStage;                            // buffers of stage st and of stage st + 3
  if (nstages > 3) copy_stage(3, far);
  mma_step(0, true, cur, 1, 0, false, 0, 0);
  const int whole = ragged_stage < 0 ? nstages : nstages - 1;    // stages whose copies take the common form
  int st = 1;
  for (; st + 3 < whole; st++) {
    cur = next_buf(cur); far = next_buf(far);
    wait_copies_and_barrier<4 * kCopies, false>();
    mma_step(1, true, cur, 0, 0, true, st + 3, far);             // the last step of stage st - 1
    mma_step(0, true, cur, 1, 1, true, st + 3, far);
  }
  for (; st < nstages; st++) {
    cur = next_buf(cur); far = next_buf(far);
    arrive(st, cur);
    if (st + 3 < nstages) copy_ragged(st + 3, far);
    mma_step(1, true, cur, 0, 0, false, 0, 0);
    mma_step(0, true, cur, 1, 0, false, 0, 0);
  }
  mma_step(1, false, 0, 0, 0, false, 0, 0);

  if (SUMS && at.tile_j == 0) {
#pragma unroll
    for (int h = 0; h < kSums; h++) {
      const float v = colsum[h] + __shfl_xor(colsum[h], 32);
      const int64_t row = i0 + fragment_row(wave, h) + l32;
      if (lh == 0) {
        if (splits > 1) sums[(int64_t)at.split * tiles_i * kTile + row] = v;
        else if (row < m) db[row] = from_float<T>(v);
      }
    }
  }
  if (splits > 1) {                                              // slab (fragment, quarter) of the tile: 4 rows of one column per lane
    float* out = partial + (int64_t)unit * (kTile * kTile) + tid * 4;
#pragma unroll
    for (int s = 0; s < kSlabs; s++) {
      const float16v& v = acc[s / (4 * kTJ)][(s >> 2) % kTJ];
      const int r = (s & 3) * 4;
      *reinterpret_cast<float4v*>(out + s * (kThreads * 4)) = float4v{v[r], v[r + 1], v[r + 2], v[r + 3]};
    }
    return;
  }
#pragma unroll
  for (int s = 0; s < kSlabs; s++) {
    const int64_t row = i0 + fragment_row(wave, s / (4 * kTJ)) + (s & 3) * 8 + lh * 4, col = j0 + (wj * kTJ + (s >> 2) % kTJ) * 32 + l32;
    if (row < m && col < n) {
#pragma unroll
      for (int r = 0; r < 4; r++) dw[(row + r) * n + col] = from_float<T>(acc[s / (4 * kTJ)][(s >> 2) % kTJ][(s & 3) * 4 + r]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// dW and db from the pieces: block (tile, slab), and with blockIdx.x one past the tiles the sums of the columns
template <typename T>
__global__ void __launch_bounds__(kThreads)
grad_weight_reduce(const float* __restrict__ partial, const float* __restrict__ sums, int splits, int64_t m, int64_t n, int tiles_i, int tiles_j,
                   T* __restrict__ dw, T* __restrict__ db) {
  const int ntiles = tiles_i * tiles_j, tid = threadIdx.x;
  if ((int)blockIdx.x == ntiles) {
    for (int64_t i = (int64_t)blockIdx.y * kThreads + tid; i < m; i += (int64_t)gridDim.y * kThreads) {
      float v = 0.0f;
      for (int p = 0; p < splits; p++) v += sums[(int64_t)p * tiles_i * kTile + i];
      db[i] = from_float<T>(v);
    }
    return;
  }
  const Piece at = locate((int)blockIdx.x, tiles_i, tiles_j);
  const int lane = tid & 63, wave = tid >> 6, s = (int)blockIdx.y;
  const int64_t row = (int64_t)at.tile_i * kTile + fragment_row(wave, s / (4 * kTJ)) + (s & 3) * 8 + (lane >> 5) * 4;
  const int64_t col = (int64_t)at.tile_j * kTile + ((wave % kWavesJ) * kTJ + (s >> 2) % kTJ) * 32 + (lane & 31);
  if (row >= m || col >= n) return;
  const float* first = partial + (int64_t)blockIdx.x * (kTile * kTile) + s * (kThreads * 4) + tid * 4;
  const int64_t piece = (int64_t)ntiles * (kTile * kTile);
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
  for (int r = 0; r < 4; r++) dw[(row + r) * n + col] = from_float<T>(v[r]);
}

int64_t piece_bytes(int64_t tiles_i, int64_t tiles_j) { return (tiles_i * tiles_j * kTile + tiles_i) * kTile * 4; }

// The number of pieces with the least  stages of one piece x 0.6 us + (more than one: 3 us + 0.32 us per MB of partial tiles),
// all in one round of the compute units.  The constants are fitted to timings of 1 to 16 pieces over 500 to 16384 tokens
// and 2048 x 512 to 6400 x 1600 outputs; the choice is within 4 % of the best on all of them.  More than 128 tiles stay in one
// piece, since two would need a second round of the compute units (against the library's product see _linear16).  36 tiles, us:
// 12288 tokens 209 in one piece, 82 in three, 72 in seven; 1024 tokens 24 in one, 31 in seven.
int choose_pieces(int64_t tokens, int64_t tiles_i, int64_t tiles_j, int64_t workspace_bytes) {
  const int64_t stages = (tokens + kStageTokens - 1) / kStageTokens, tiles = tiles_i * tiles_j;
  int best = 1;
  double least = (double)stages * 0.6;
  for (int64_t p = 2; p <= kMaxPieces && p <= stages / 4 && p * tiles <= 256 && p * piece_bytes(tiles_i, tiles_j) <= workspace_bytes; p++) {
    const double us = (double)((stages + p - 1) / p) * 0.6 + 3.0 + (double)(p * tiles) * (kTile * kTile * 4e-6 * 0.32);
    if (us < least) { least = us; best = (int)p; }
  }
  return best;
}

template <typename T>
int launch(const void* g, int64_t ldg, const void* x, int64_t ldx, int64_t tokens, int64_t m, int64_t n, void* dw, void* db,
           void* workspace, int64_t workspace_bytes, hipStream_t s) {
  const int tiles_i = (int)((m + kTile - 1) / kTile), tiles_j = (int)((n + kTile - 1) / kTile);
  const int pieces = workspace ? choose_pieces(tokens, tiles_i, tiles_j, workspace_bytes) : 1;
  float* partial = (float*)workspace;
  float* sums = pieces > 1 ? partial + (int64_t)pieces * tiles_i * tiles_j * kTile * kTile : nullptr;     // behind the partial tiles
  const int per_xcd = (tiles_i * tiles_j * pieces + 7) / 8;
  auto pipe = [&](auto with_sums) {
    hipLaunchKernelGGL((grad_weight_pipe<T, decltype(with_sums)::value>), dim3((unsigned)(per_xcd * 8)), dim3(kThreads), 0, s, (const uint8_t*)g, ldg * 2,
                       (const uint8_t*)x, ldx * 2, tokens, m, n, tiles_i, tiles_j, pieces, partial, sums, (T*)dw, (T*)db);
  };
  if (db) pipe(std::true_type{}); else pipe(std::false_type{});
  if (pieces > 1)
    hipLaunchKernelGGL((grad_weight_reduce<T>), dim3((unsigned)(tiles_i * tiles_j + (db ? 1 : 0)), kSlabs), dim3(kThreads), 0, s, partial, sums, pieces, m, n,
                       tiles_i, tiles_j, (T*)dw, (T*)db);
  return check_launch("tf24_grad_weight");
}

}  // namespace
}  // namespace tf24

extern "C" int64_t tf24_grad_weight_workspace_bytes(int64_t tokens, int64_t m, int64_t n) {
  using namespace tf24;
  if (tokens <= 0 || m <= 0 || n <= 0) return 0;
  const int64_t tiles_i = (m + kTile - 1) / kTile, tiles_j = (n + kTile - 1) / kTile;
  const int pieces = choose_pieces(tokens, tiles_i, tiles_j, (int64_t)1 << 40);
  return pieces > 1 ? pieces * piece_bytes(tiles_i, tiles_j) : 0;
}

extern "C" int tf24_grad_weight(const void* g, int64_t ldg, const void* x, int64_t ldx, int dtype, int64_t tokens, int64_t m, int64_t n,
                                void* dw, void* db, void* workspace, int64_t workspace_bytes, void* stream) {
  using namespace tf24;
  const char* fn = "tf24_grad_weight";
  if (dtype != TF24_F16 && dtype != TF24_BF16) return fail(TF24_ERR_DTYPE, "%s: unsupported dtype %d", fn, dtype);
  if (tokens <= 0 || tokens > 0x7fffffffLL) return fail(TF24_ERR_SHAPE, "%s: bad number of tokens %lld", fn, (long long)tokens);
  if (m <= 0 || m % 8 || n <= 0 || n % 8 || m > (1 << 20) || n > (1 << 20))
    return fail(TF24_ERR_SHAPE, "%s: %lld x %lld must be positive multiples of 8, at most %d", fn, (long long)m, (long long)n, 1 << 20);
  // 32 tokens are addressed by 32-bit lane offsets
  if (ldg < m || ldg % 8 || ldg > (1 << 23) || ldx < n || ldx % 8 || ldx > (1 << 23))
    return fail(TF24_ERR_STRIDE, "%s: leading dimensions %lld, %lld must cover the rows, be multiples of 8 and at most %d", fn, (long long)ldg, (long long)ldx, 1 << 23);
  if (!g || !x || !dw) return fail(TF24_ERR_ARG, "%s: null pointer", fn);
  if (workspace_bytes < 0) return fail(TF24_ERR_ARG, "%s: negative workspace size", fn);
  if (int rc = check_aligned(fn, 16, {g, x, workspace})) return rc;
  if (int rc = check_aligned(fn, 2, {dw, db})) return rc;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == TF24_F16) return launch<f16_t>(g, ldg, x, ldx, tokens, m, n, dw, db, workspace, workspace_bytes, s);
  return launch<bf16_t>(g, ldg, x, ldx, tokens, m, n, dw, db, workspace, workspace_bytes, s);
}
