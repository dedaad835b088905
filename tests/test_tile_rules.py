"""The rules by which a product chooses its tiles, called on the CPU as the launch code calls them."""
import ctypes
import importlib.util
import os
import subprocess

import pytest

from test_gpu_parity import SQUARE, STAGE_ORDER

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
extern "C" int rotate_from() { return tf24::kRotateMinStages; }
""")
    subprocess.run([build.HIPCC, *build.FLAGS, "--offload-host-only", "-shared", str(src), "-o", str(lib)], check=True, capture_output=True)
    handle = ctypes.CDLL(str(lib))
    handle.square.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_int]
    handle.tiles.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_int]
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
