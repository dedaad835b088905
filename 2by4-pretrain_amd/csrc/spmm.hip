// tf24_spmm: argument checks and dispatch on the operand type.  The kernels live in spmm_kernels.hpp and are
// instantiated by one translation unit per operand type (spmm_f16.hip, spmm_bf16.hip, spmm_e4m3.hip,
// spmm_e5m2.hip, spmm_i8.hip), so that they compile side by side.
#include "spmm_kernels.hpp"

namespace tf24 {
namespace {
// extent: what the number of dense columns must be a multiple of (0: the operand type's own)
int validate(const char* fn, int dtype, int64_t n_sparse, int64_t k, int b_layout, int64_t ldb, int64_t n_dense, int64_t extent,
             int out_dtype, int c_layout, int64_t ldc, int activation) {
  const bool bias_f32 = activation & TF24_BIAS_F32;
  activation &= ~TF24_BIAS_F32;
  if (dtype != TF24_F16 && dtype != TF24_BF16 && !is_8bit(dtype)) return fail(TF24_ERR_DTYPE, "%s: unsupported operand dtype %d", fn, dtype);
  if (dtype == TF24_I8) {
    // integer product (.cu:594-637): int32 results, no or ReLU activation
    if (out_dtype != TF24_I32) return fail(TF24_ERR_DTYPE, "%s: int8 operands give int32 results (output dtype %d)", fn, out_dtype);
    if (activation != TF24_ACT_NONE && activation != TF24_ACT_RELU) return fail(TF24_ERR_ARG, "%s: int8 operands support no activation or ReLU (%d)", fn, activation);
  } else if (out_dtype != TF24_F16 && out_dtype != TF24_BF16 && out_dtype != TF24_F32) {
    return fail(TF24_ERR_DTYPE, "%s: unsupported output dtype %d", fn, out_dtype);
  }
  const bool eight = is_8bit(dtype);
  const int64_t kmult = eight ? 128 : 64, dmult = eight ? 16 : 8;
  if (n_sparse <= 0 || n_sparse % 32) return fail(TF24_ERR_SHAPE, "%s: sparse operand rows %lld must be a positive multiple of 32", fn, (long long)n_sparse);
  if (k <= 0 || k % kmult) return fail(TF24_ERR_SHAPE, "%s: inner dimension %lld must be a positive multiple of %lld", fn, (long long)k, (long long)kmult);
  if (n_dense <= 0 || n_dense % (extent ? extent : dmult)) return fail(TF24_ERR_SHAPE, "%s: dense operand extent %lld must be a positive multiple of %lld", fn, (long long)n_dense, (long long)(extent ? extent : dmult));
  if (b_layout != TF24_ROW_MAJOR && b_layout != TF24_COL_MAJOR) return fail(TF24_ERR_ARG, "%s: bad b_layout %d", fn, b_layout);
  if (c_layout != TF24_ROW_MAJOR && c_layout != TF24_COL_MAJOR) return fail(TF24_ERR_ARG, "%s: bad c_layout %d", fn, c_layout);
  const int64_t bext = b_layout == TF24_ROW_MAJOR ? k : n_dense;
  if (ldb < bext || ldb % dmult) return fail(TF24_ERR_STRIDE, "%s: ldb %lld must be >= %lld and a multiple of %lld", fn, (long long)ldb, (long long)bext, (long long)dmult);
  // the copies address a tile's rows of B by 32-bit lane offsets from the tile's base: 256 rows must span < 4 GiB
  if (ldb * (eight ? 1 : 2) > ((int64_t)1 << 24)) return fail(TF24_ERR_STRIDE, "%s: ldb %lld exceeds 16 MiB per row", fn, (long long)ldb);
  const int64_t cext = c_layout == TF24_ROW_MAJOR ? n_dense : n_sparse;
  // rows of the output leave as 16-byte stores: 8 elements of a 16-bit type, 4 of a 32-bit one
  const int64_t cmult = (out_dtype == TF24_F16 || out_dtype == TF24_BF16) ? 8 : 4;
  if (ldc < cext || ldc % cmult) return fail(TF24_ERR_STRIDE, "%s: ldc %lld must be >= %lld and a multiple of %lld", fn, (long long)ldc, (long long)cext, (long long)cmult);
  if (activation < TF24_ACT_NONE || activation > TF24_ACT_GELU) return fail(TF24_ERR_ARG, "%s: bad activation %d", fn, activation);
  if (bias_f32 && out_dtype == TF24_I32) return fail(TF24_ERR_ARG, "%s: integer results take an integer bias", fn);
  return TF24_OK;
}
}  // namespace
}  // namespace tf24

extern "C" int tf24_spmm_validate(int dtype, int64_t n_sparse, int64_t k, int b_layout, int64_t ldb, int64_t n_dense,
                                  int out_dtype, int c_layout, int64_t ldc, int activation) {
  return tf24::validate("tf24_spmm", dtype, n_sparse, k, b_layout, ldb, n_dense, 0, out_dtype, c_layout, ldc, activation);
}

namespace tf24 {
namespace {
// the float32 partial tiles of the pieces chosen with any workspace
template <typename T, typename C>
int64_t piece_bytes(int64_t n_sparse, int64_t k, int64_t n_dense, bool k_strided) {
  const int pieces = choose_pieces<T, C>(n_sparse, k, n_dense, (int64_t)1 << 40, k_strided).count;
  if (pieces < 2) return 0;
  return pieces * ((n_sparse + C::BI - 1) / C::BI) * ((n_dense + C::BJ - 1) / C::BJ) * C::BI * C::BJ * 4;
}
// for either orientation of the dense operand that the kernels of this operand size take (dispatch_out)
template <typename T>
int64_t workspace_bytes(int64_t n_sparse, int64_t k, int64_t n_dense) {
  const int64_t strided = sizeof(T) == 2 && n_dense % 8 == 0 ? std::max(piece_bytes<T, TiledCfg>(n_sparse, k, n_dense, true),
                                                                       piece_bytes<T, SquareCfg>(n_sparse, k, n_dense, true)) : 0;
  if (n_dense <= narrow_columns(n_sparse, k * (int64_t)sizeof(T) / 128, sizeof(T) == 1)) return strided;
  // (for weights of 129 to 168 rows of 128 x 64 tiles the scratch of the 256 x 64 ones from 64 stages on, also where the product is the faster in one
  // piece of the former and leaves it alone: sizes that programs hold for a weight stay what they were)
  const int64_t rows = (n_sparse + SlimCfg::BI - 1) / SlimCfg::BI, stages = k * (int64_t)sizeof(T) / SlimCfg::KB;
  if (n_dense <= SlimCfg::BJ && rows > 128 && rows <= 168 && stages >= 64) return std::max(strided, piece_bytes<T, TallSlimCfg>(n_sparse, k, n_dense, false));
  const bool tall_slim = n_dense <= SlimCfg::BJ && takes_tall_slim(n_sparse, stages, sizeof(T) == 1);
  return std::max(strided, tall_slim ? piece_bytes<T, TallSlimCfg>(n_sparse, k, n_dense, false)
                           : n_dense <= SlimCfg::BJ ? piece_bytes<T, SlimCfg>(n_sparse, k, n_dense, false)
                           : takes_small<T>(n_sparse, k, n_dense, (int64_t)1 << 40) ? piece_bytes<T, SmallCfg>(n_sparse, k, n_dense, false)
                           : takes_mid<T>(n_sparse, k, n_dense, (int64_t)1 << 40) ? piece_bytes<T, MidCfg>(n_sparse, k, n_dense, false)
                                                                                  : piece_bytes<T, TiledCfg>(n_sparse, k, n_dense, false));
}
}  // namespace
}  // namespace tf24

extern "C" int64_t tf24_spmm_workspace_bytes(int dtype, int64_t n_sparse, int64_t k, int64_t n_dense) {
  using namespace tf24;
  return is_8bit(dtype) ? workspace_bytes<e4m3_t>(n_sparse, k, n_dense) : workspace_bytes<f16_t>(n_sparse, k, n_dense);
}

namespace tf24 {
namespace {
int run_spmm(const char* fn, const void* a_values, const void* a_meta, int a_layout, int dtype, int64_t n_sparse, int64_t k,
             const void* b, int b_layout, int64_t ldb, int64_t n_dense, int64_t extent, void* c, int out_dtype, int c_layout, int64_t ldc,
             const void* bias, float scale, int activation, void* workspace, int64_t workspace_bytes, void* stream, RowSums* sums = nullptr) {
  const int bias_f32 = activation & TF24_BIAS_F32;
  int rc = validate(fn, dtype, n_sparse, k, b_layout, ldb, n_dense, extent, out_dtype, c_layout, ldc, activation);
  if (rc) return rc;
  if (!a_values || !a_meta || !b || !c) return fail(TF24_ERR_ARG, "%s: null pointer", fn);
  if ((rc = check_aligned(fn, 16, {a_values, b, c, workspace}))) return rc;
  // panel metadata is copied 16 bytes per lane; canonical metadata is read in words of up to 4 bytes, row pitch k/8
  if ((rc = check_aligned(fn, a_layout == TF24_COMPRESSED_PANEL ? 16 : a_layout == TF24_COMPRESSED_CUTLASS ? 4 : 8, {a_meta}))) return rc;
  if ((rc = check_aligned(fn, bias_f32 ? 4 : dtype_size(out_dtype), {bias}))) return rc;
  if (a_layout != TF24_COMPRESSED_CANONICAL && a_layout != TF24_COMPRESSED_PANEL && a_layout != TF24_COMPRESSED_CUTLASS)
    return fail(TF24_ERR_ARG, "%s: bad compressed layout %d", fn, a_layout);
  hipStream_t s = (hipStream_t)stream;
  if (dtype == TF24_I8 && scale != 1.0f) return fail(TF24_ERR_ARG, "%s: int8 products are exact, scale must be 1 (%g given)", fn, (double)scale);
  switch (dtype) {
    case TF24_I8: return spmm_i8(out_dtype, a_values, a_meta, a_layout, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, activation, workspace, workspace_bytes, s, sums);
    case TF24_F16: return spmm_f16(out_dtype, a_values, a_meta, a_layout, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, activation, workspace, workspace_bytes, s, sums);
    case TF24_BF16: return spmm_bf16(out_dtype, a_values, a_meta, a_layout, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, activation, workspace, workspace_bytes, s, sums);
    case TF24_E5M2: return spmm_e5m2(out_dtype, a_values, a_meta, a_layout, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, activation, workspace, workspace_bytes, s, sums);
    default: return spmm_e4m3(out_dtype, a_values, a_meta, a_layout, n_sparse, k, b, b_layout, ldb, n_dense, c, c_layout, ldc, bias, scale, activation, workspace, workspace_bytes, s, sums);
  }
}
}  // namespace
}  // namespace tf24

extern "C" int tf24_spmm(const void* a_values, const void* a_meta, int a_layout, int dtype, int64_t n_sparse, int64_t k,
                         const void* b, int b_layout, int64_t ldb, int64_t n_dense,
                         void* c, int out_dtype, int c_layout, int64_t ldc,
                         const void* bias, float scale, int activation, void* workspace, int64_t workspace_bytes, void* stream) {
  return tf24::run_spmm("tf24_spmm", a_values, a_meta, a_layout, dtype, n_sparse, k, b, b_layout, ldb, n_dense, 0, c, out_dtype, c_layout, ldc,
                        bias, scale, activation, workspace, workspace_bytes, stream);
}

// Rows of x are the dense columns with k contiguous, rows of y the output stored j-major: in that orientation no kernel
// loads or stores more than one row of either with one access, rows past the last are clamped on loads and skipped on
// stores, so any number of rows goes (in the other orientations 16-byte accesses run along the dense columns).
// A copy padded to a multiple of 8 rows costs what it moves: 3001 x 11008 bf16 36 us beside a product of 131 us, one row of
// 4096 two launches of 3.5 us beside one of 13 us.
extern "C" int tf24_linear(const void* a_values, const void* a_meta, int a_layout, int dtype, int64_t n_sparse, int64_t k,
                           const void* x, int64_t ldx, int64_t rows, void* y, int out_dtype, int64_t ldy,
                           const void* bias, float scale, int activation, void* workspace, int64_t workspace_bytes, void* stream) {
  return tf24::run_spmm("tf24_linear", a_values, a_meta, a_layout, dtype, n_sparse, k, x, TF24_ROW_MAJOR, ldx, rows, 1, y, out_dtype,
                        TF24_COL_MAJOR, ldy, bias, scale, activation, workspace, workspace_bytes, stream);
}

// ---- the weight gradient of the transposable layer: MVUE24(dY^T) . X and the row sums of dY^T, three launches and one workspace: conversion, product in
// pieces of the token axis, their sum with the row sums; of a product in one piece the row sums are the third launch (some 4 us).
namespace tf24 {
namespace {
struct GradSpace { int64_t meta, partial, pieces, pieces_bytes, total; };          // offsets behind the compressed values
GradSpace grad_space(int64_t m, int64_t n, int64_t tokens) {
  auto up = [](int64_t b) { return (b + 255) / 256 * 256; };
  GradSpace g;
  g.meta = up(m * tokens);                                                          // (two bytes for every other element)
  g.partial = g.meta + up(m * tokens / 8);
  g.pieces = g.partial + up(tf24_prune_compress_rowsum_workspace_bytes(m, tokens));
  g.pieces_bytes = tf24_spmm_workspace_bytes(TF24_F16, m, tokens, n);
  g.total = g.pieces + g.pieces_bytes;
  return g;
}
}  // namespace
}  // namespace tf24

extern "C" int64_t tf24_mvue_weight_grad_workspace_bytes(int64_t m, int64_t n, int64_t tokens) {
  return m > 0 && n > 0 && tokens > 0 ? tf24::grad_space(m, n, tokens).total : 0;
}

extern "C" int tf24_mvue_weight_grad(const void* grad, int64_t ldg, const void* x, int64_t ldx, int dtype, int64_t m, int64_t n, int64_t tokens, int mode,
                                     const void* rnd, void* dw, int dw_dtype, void* db, int db_dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  using namespace tf24;
  const char* fn = "tf24_mvue_weight_grad";
  if (dtype != TF24_F16 && dtype != TF24_BF16) return fail(TF24_ERR_DTYPE, "%s: unsupported operand dtype %d", fn, dtype);
  if (db_dtype != TF24_F32 && db_dtype != TF24_F16 && db_dtype != TF24_BF16) return fail(TF24_ERR_DTYPE, "%s: unsupported row-sum dtype %d", fn, db_dtype);
  if (mode != TF24_PRUNE_MVUE_SEEDED && mode != TF24_PRUNE_MVUE_SEEDED_DEVICE) return fail(TF24_ERR_ARG, "%s: mode %d does not draw its uniforms", fn, mode);
  // (everything that the product will ask for, before the conversion is launched)
  int rc = validate(fn, dtype, m, tokens, TF24_COL_MAJOR, ldx, n, 0, dw_dtype, TF24_ROW_MAJOR, n, TF24_ACT_NONE);
  if (rc) return rc;
  if (!grad || !x || !dw || !db || !workspace) return fail(TF24_ERR_ARG, "%s: null pointer", fn);
  const GradSpace at = grad_space(m, n, tokens);
  if (workspace_bytes < at.total)
    return fail(TF24_ERR_ARG, "%s: workspace of %lld bytes is too small (%lld needed)", fn, (long long)workspace_bytes, (long long)at.total);
  if ((rc = check_aligned(fn, 16, {x, dw, workspace}))) return rc;
  if ((rc = check_aligned(fn, dtype_size(db_dtype), {db}))) return rc;
  uint8_t* const ws = (uint8_t*)workspace;
  float* const partial = (float*)(ws + at.partial);
  if ((rc = compress_with_partial_sums(fn, grad, dtype, ldg, m, tokens, mode, rnd, ws, ws + at.meta, partial, (hipStream_t)stream))) return rc;
  RowSums sums{partial, (int)((tokens + 127) / 128), m, db, db_dtype};
  rc = run_spmm(fn, ws, ws + at.meta, TF24_COMPRESSED_PANEL, dtype, m, tokens, x, TF24_COL_MAJOR, ldx, n, 0, dw, dw_dtype, TF24_ROW_MAJOR, n, nullptr, 1.0f, TF24_ACT_NONE,
                at.pieces_bytes ? ws + at.pieces : nullptr, at.pieces_bytes, stream, &sums);
  return rc || !sums.partial ? rc : finish_row_sums(fn, sums, (hipStream_t)stream);
}
