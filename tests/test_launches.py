"""What a product launches, on the CPU: the launch code of spmm_kernels.hpp with launches that are written down instead of made."""
import ctypes
import importlib.util
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    spec = importlib.util.spec_from_file_location("tf24_build", os.path.join(ROOT, "2by4-pretrain_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    folder = tmp_path_factory.mktemp("launches")
    src, lib = folder / "launches.hip", folder / "launches.so"
    src.write_text("""
#include <hip/hip_runtime.h>
#include <string>
static std::string made;                                 // the kernels launched, one a line
#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(kernel, grid, block, ...) (made += std::string(#kernel) + "\\n", (void)(grid), (void)(block))
#include "spmm_kernels.hpp"
namespace tf24 {
int check_launch(const char*) { return 0; }
}
// a float16 product with row-major results and row sums to finish; returns whether its launches finish them
template <typename C>
static int with_sums(int64_t n_sparse, int64_t n_dense, int64_t stages, int b_layout, int64_t scratch) {
  made.clear();
  tf24::RowSums sums{(const float*)256, 1, n_sparse, (void*)256, TF24_F32};
  tf24::launch_tiled<tf24::f16_t, tf24::f16_t, C>((void*)256, (void*)256, n_sparse, stages * 64, (void*)256, b_layout, b_layout == TF24_ROW_MAJOR ? stages * 64 : n_dense, n_dense,
                                                  (void*)256, TF24_ROW_MAJOR, n_dense, nullptr, 1.0f, 0, scratch ? (void*)256 : nullptr, scratch, nullptr, &sums);
  return !sums.partial;
}
extern "C" int small_with_sums(int64_t n, int64_t j, int64_t stages, int64_t scratch) { return with_sums<tf24::SmallCfg>(n, j, stages, TF24_ROW_MAJOR, scratch); }
extern "C" int mid_with_sums(int64_t n, int64_t j, int64_t stages, int64_t scratch) { return with_sums<tf24::MidCfg>(n, j, stages, TF24_ROW_MAJOR, scratch); }
extern "C" int wide_with_sums(int64_t n, int64_t j, int64_t stages, int64_t scratch) { return with_sums<tf24::TiledCfg>(n, j, stages, TF24_COL_MAJOR, scratch); }
extern "C" const char* launched() { return made.c_str(); }
""")
    res = subprocess.run([build.HIPCC, *build.FLAGS, "--offload-host-only", "-shared", str(src), "-o", str(lib)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-3000:]
    handle = ctypes.CDLL(str(lib))
    for f in (handle.small_with_sums, handle.mid_with_sums, handle.wide_with_sums):
        f.argtypes = [ctypes.c_int64] * 4
    handle.launched.restype = ctypes.c_char_p
    return handle


@pytest.mark.parametrize("tiles,n,columns,stages,scratch,pieces", [
    ("wide", 768, 3072, 192, 1 << 40, True), ("wide", 768, 3072, 192, 0, False),
    ("small", 1184, 136, 30, 1 << 40, True), ("small", 1184, 136, 30, 0, False),
    ("mid", 1184, 136, 100, 1 << 40, True)])
def test_a_product_in_pieces_is_added_whoever_finishes_the_row_sums(launches, tiles, n, columns, stages, scratch, pieces):
    """Every product in pieces launches their sum, whatever its tiles; the row sums that come with it are finished there or left to the caller."""
    finished = getattr(launches, tiles + "_with_sums")(n, columns, stages, scratch)
    made = launches.launched().decode().splitlines()
    assert ["spmm_reduce_splits" in line for line in made] == ([False, True] if pieces else [False]), made
    assert finished == (pieces and tiles == "wide")
