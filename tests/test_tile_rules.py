"""The rules by which a product chooses its tiles, called on the CPU as the launch code calls them."""
import ctypes
import importlib.util
import os
import subprocess

import pytest

from test_gpu_parity import NOT_TALL, SQUARE, SQUARE_STRIDED, STAGE_ORDER, TALL

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CU_SLOTS = 32                      # compute units of an XCD


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    spec = importlib.util.spec_from_file_location("tf24_build", os.path.join(ROOT, "2by4-pretrain_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    folder = tmp_path_factory.mktemp("rules")
    src, lib = folder / "rules.hip", folder / "rules.so"
    src.write_text("""
#include "spmm_kernels.hpp"
extern "C" int square(int64_t n_sparse, int64_t n_dense, int stages, int cu_slots) {
  return tf24::takes_square(n_sparse, n_dense, stages, tf24::full_rounds(n_sparse, n_dense, stages, cu_slots), cu_slots);
}
extern "C" int tiles(int64_t n_sparse, int64_t n_dense, int stages, int results16, int cu_slots) {
  const tf24::TileRows rows = tf24::full_rounds(n_sparse, n_dense, stages, cu_slots);
  return (int)tf24::choose_tiles(n_sparse, n_dense, stages, rows, results16, cu_slots) + (rows.tail_rows ? 100 : 0);
}
extern "C" int strided(int64_t n_sparse, int64_t n_dense, int stages, int results16, int jmajor, int cu_slots) {
  auto* rule = results16 ? tf24::strided_takes_square<tf24::f16_t, tf24::f16_t> : tf24::strided_takes_square<tf24::f16_t, float>;
  return rule(n_sparse, (int64_t)stages * 64, n_dense, (int64_t)1 << 40, jmajor, cu_slots);
}
extern "C" int strided_pieces(int64_t n_sparse, int64_t n_dense, int stages) {
  return tf24::choose_pieces<tf24::f16_t, tf24::SquareCfg>(n_sparse, (int64_t)stages * 64, n_dense, (int64_t)1 << 40, true).count;
}
extern "C" int tiles_of_16_bits(int64_t n_sparse, int64_t n_dense, int stages, int cu_slots) {
  const tf24::TileRows rows = tf24::full_rounds(n_sparse, n_dense, stages, cu_slots);
  return (int)tf24::choose_tiles(n_sparse, n_dense, stages, rows, true, cu_slots, true) + (rows.tail_rows ? 100 : 0);
}
extern "C" int rotate_from() { return tf24::kRotateMinStages; }
""")
    subprocess.run([build.HIPCC, *build.FLAGS, "--offload-host-only", "-shared", str(src), "-o", str(lib)], check=True, capture_output=True)
    handle = ctypes.CDLL(str(lib))
    handle.square.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_int]
    handle.tiles.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_int]
    handle.tiles_of_16_bits.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_int]
    handle.strided.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int]
    handle.strided_pieces.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    return handle


@pytest.mark.parametrize("n,stages,columns,square", [
    # measured 5 % or more apart (us on the other tiles, on square ones); below 32 stages the other tiles are 8-wave ones
    (3072, 12, 12288, 0), (3072, 12, 8192, 0), (2304, 12, 12288, 0),          # 44.2 48.3, 30.1 33.6, 32.7 37.2
    (2048, 8, 12288, 0), (6400, 25, 4096, 0), (6656, 11, 12879, 0),           # 23.9 27.9, 53.3 59.8, 86.2 101.4
    (8576, 41, 3066, 0), (3072, 128, 8536, 0), (11008, 64, 4096, 0),          # 76.9 80.3, 232 250, 185 205
    (4096, 15, 4145, 1), (4320, 25, 7701, 1)])                                # 31.9 26.4, 75.1 70.6
def test_square_tiles_where_they_are_the_faster_ones(rules, n, stages, columns, square):
    assert rules.square(n, columns, stages, CU_SLOTS) == square


@pytest.mark.parametrize("n,stages,rows,tiles,rotates", STAGE_ORDER + [case[:3] + ("square",) + case[3:] for case in SQUARE])
def test_products_tested_on_the_gpu_take_the_tiles_they_are_for(rules, n, stages, rows, tiles, rotates):
    code = rules.tiles(n, rows, stages, 1, CU_SLOTS)
    assert code == {"wide": 1, "wide, two launches": 101, "narrow": 2, "square": 3}[tiles]
    assert rotates == (stages >= rules.rotate_from())
    # more than one round of half tiles, which would be taken first, and no room for pieces of k
    assert -(-n // 256) * -(-rows // 128) > 256 and -(-n // 256) * -(-rows // 256) > 128


@pytest.mark.parametrize("n,stages,columns,pieces", SQUARE_STRIDED)
def test_k_strided_products_tested_on_the_gpu_take_square_tiles(rules, n, stages, columns, pieces):
    assert rules.strided_pieces(n, columns, stages) == pieces
    # with float32 results and with 16-bit ones stored j-major; i-major ones only where a reduction writes them
    forms = [rules.strided(n, columns, stages, results16, jmajor, CU_SLOTS) for results16, jmajor in ((0, 0), (1, 1), (1, 0))]
    assert forms == [1, 1, int(pieces > 1)]


@pytest.mark.parametrize("n,stages,columns,tall", [
    # measured apart (us on the other tiles, on 384 x 192 ones)
    (1120, 44, 14480, 1), (1504, 30, 11707, 1), (2912, 91, 12074, 1), (11008, 64, 8192, 1),            # 69.9 54.8, 53.1 42.3, 244 200, 358 346
    (8192, 128, 8192, 0), (5280, 12, 8114, 0), (1312, 161, 13869, 0), (11776, 35, 1599, 0)]            # 497 518, 46.8 59.5, 231 288, 54.3 70.4
    + [(n, stages, rows, 1) for n, stages, rows, _ in TALL])
def test_tall_tiles_where_they_are_the_faster_ones(rules, n, stages, columns, tall):
    assert (rules.tiles_of_16_bits(n, columns, stages, CU_SLOTS) % 100 == 4) == tall


@pytest.mark.parametrize("n,stages,rows,tiles", NOT_TALL)
def test_other_tiles_are_tested_with_16_bits_too(rules, n, stages, rows, tiles):
    assert rules.tiles_of_16_bits(n, rows, stages, CU_SLOTS) == {"wide, two launches": 101, "square": 3}[tiles]
