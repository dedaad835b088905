"""What a product launches, on the CPU: the launch code of spmm_kernels.hpp with launches that are written down instead of made."""
import ctypes
import importlib.util
import os
import subprocess

import pytest

from test_gpu_parity import MID_PIECES, SLIM_TILES, TALL_SLIM_TILES

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
struct C { static constexpr int BI = 0, BJ = 0; };        // for launches outside of a function that has tiles of that name
#define hipLaunchKernelGGL(kernel, grid, block, ...) \\
  (made += std::string(#kernel) + " " + std::to_string(C::BI) + "x" + std::to_string(C::BJ) + "\\n", (void)(grid), (void)(block))
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
// the product of a weight of n rows and j rows of activations (linear), its scratch as asked for
template <typename T>
static void linear(int64_t n, int64_t j, int64_t stages) {
  const int64_t k = stages * 128 / (int64_t)sizeof(T);
  tf24::dispatch_out<T>(TF24_F16, (void*)256, (void*)256, TF24_COMPRESSED_PANEL, n, k, (void*)256, TF24_ROW_MAJOR, k, j, (void*)256, TF24_COL_MAJOR, n, nullptr, 1.0f, 0, (void*)256,
                        (int64_t)1 << 40, nullptr, nullptr);
}
extern "C" void product(int bytes, int64_t n, int64_t j, int64_t stages) {
  made.clear();
  if (bytes == 1) linear<tf24::e4m3_t>(n, j, stages);
  else linear<tf24::f16_t>(n, j, stages);
}
extern "C" int waves(int64_t blocks, int64_t panels, int64_t columns) { return tf24::few_waves(blocks, panels, columns); }
extern "C" const char* launched() { return made.c_str(); }
""")
    res = subprocess.run([build.HIPCC, *build.FLAGS, "--offload-host-only", "-shared", str(src), "-o", str(lib)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-3000:]
    handle = ctypes.CDLL(str(lib))
    for f in (handle.small_with_sums, handle.mid_with_sums, handle.wide_with_sums):
        f.argtypes = [ctypes.c_int64] * 4
    handle.product.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3
    handle.waves.argtypes = [ctypes.c_int64] * 3
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


def kernels_of(launches, size, n, columns, stages):
    """The names of the kernels that such a product launches, tiles by their rows and columns."""
    launches.product(size, n, columns, stages)
    return [line[1:line.index("<")] + line[line.rindex(" "):].replace(" 0x0", "") for line in launches.launched().decode().splitlines()]


@pytest.mark.parametrize("size,n,panels,columns,kernel", [
    # us before spmm_few, on it, and on spmm_narrow again
    (2, 256, 4, 16, "spmm_narrow"), (2, 2144, 4, 16, "spmm_narrow"), (1, 864, 3, 16, "spmm_narrow"), (1, 928, 6, 16, "spmm_narrow"),      # 2.88 3.36 2.88, 3.13 3.42 3.13, 3.04 3.42 3.04, 3.14 3.49 3.15
    (2, 4096, 7, 9, "spmm_narrow"), (2, 6016, 4, 14, "spmm_narrow"), (1, 4832, 5, 16, "spmm_narrow"),                                    # 3.3 3.7 3.3 (from the caches)
    (2, 256, 4, 8, "spmm_few"), (2, 2144, 8, 16, "spmm_few"), (2, 8224, 4, 16, "spmm_few"), (2, 4096, 28, 32, "spmm_few"), (2, 2304, 11, 32, "spmm_narrow")])
def test_short_products_of_few_columns(launches, size, n, panels, columns, kernel):
    assert kernels_of(launches, size, n, columns, panels) == [kernel]


@pytest.mark.parametrize("panels,columns,blocks,waves", [
    # one chunk of four panels holds a wave's share from 17 columns on, up to the most waves
    (12, 17, 192, 4), (16, 32, 192, 4), (17, 26, 192, 8), (23, 25, 256, 8), (24, 32, 256, 8), (64, 32, 256, 8), (17, 24, 300, 4), (32, 32, 512, 4), (12, 20, 257, 4),
    (12, 1, 192, 2), (24, 16, 192, 4), (48, 8, 256, 8), (64, 1, 384, 4), (128, 1, 512, 2), (64, 8, 688, 2)])
def test_waves_that_share_a_row_block(launches, panels, columns, blocks, waves):
    assert launches.waves(blocks, panels, columns) == waves


@pytest.mark.parametrize("n,panels,columns,kernel", [
    # e4m3 values of more than one row block a compute unit: us on spmm_narrow and on 128 x 64 tiles
    (7520, 30, 19, "spmm_narrow"), (6496, 24, 20, "spmm_narrow"), (5056, 32, 24, "spmm_narrow"),      # 8.9 11.6, 8.6 9.7, 9.4 9.6
    (5728, 19, 30, "spmm_pipe 128x64"), (5728, 33, 20, "spmm_pipe 128x64"),                            # 8.4 7.7
    (5728, 16, 30, "spmm_few"), (8224, 12, 17, "spmm_pipe 128x64"), (3008, 17, 30, "spmm_few")])
def test_8_bit_products_of_17_to_32_columns(launches, n, panels, columns, kernel):
    assert kernels_of(launches, 1, n, columns, panels)[0] == kernel


@pytest.mark.parametrize("n,stages,columns", MID_PIECES)
def test_products_tested_on_the_gpu_take_256_x_128_tiles_in_pieces(launches, n, stages, columns):
    for size in (1, 2):
        assert kernels_of(launches, size, n, columns, stages) == ["spmm_pipe 256x128", "spmm_reduce_splits 256x128"]


@pytest.mark.parametrize("n,stages,columns", TALL_SLIM_TILES)
def test_products_tested_on_the_gpu_take_the_tall_tiles(launches, n, stages, columns):
    for size in (1, 2):
        assert kernels_of(launches, size, n, columns, stages) == ["spmm_pipe 256x64"] + ["spmm_reduce_splits 256x64"] * (n < 32768)


@pytest.mark.parametrize("size,n,stages,tall", [
    # us on 128 x 64 and on 256 x 64 tiles
    (2, 16416, 64, 0), (2, 20480, 128, 0), (1, 20480, 64, 0), (2, 32000, 64, 0), (1, 28480, 65, 0), (2, 28544, 63, 0),    # 23.7 25.9, 43.5 46.0, 31.4 46.1, 25.7 40.1
    (2, 16416, 128, 1), (2, 18880, 224, 1), (2, 16416, 102, 1), (2, 16416, 101, 0), (2, 16384, 256, 0),                  # 43.3 38.5, 77.9 63.0
    (2, 21504, 200, 1), (2, 21536, 512, 0),                                                                              # three pieces, two
    (2, 32832, 79, 1), (1, 34560, 87, 1), (2, 62592, 12, 1), (2, 47584, 3, 0), (2, 50304, 12, 1), (2, 65536, 11, 0),      # 58.2 53.7, 67.2 56.5, 15.6 13.9, 5.9 6.5
    (2, 73984, 33, 0), (1, 114976, 12, 0), (2, 114976, 5, 1), (2, 128256, 32, 1), (2, 151936, 64, 0), (2, 247104, 5, 1)])  # 13.4 11.4, 63.9 59.0, 28.7 25.3
def test_tiles_of_64_columns_of_tall_weights(launches, size, n, stages, tall):
    made = kernels_of(launches, size, n, 64, stages)
    assert made[0] == ("spmm_pipe 256x64" if tall else "spmm_pipe 128x64")
    if tall and n <= 21504:
        assert made[1:] == ["spmm_reduce_splits 256x64"]                     # in pieces, which is what these tiles are for
    elif n >= 16416:
        assert len(made) == 1


@pytest.mark.parametrize("size,n,stages,columns,tiles", [
    # us with the operands from memory on the tiles that k is cut for, on 128 x 128 ones in one piece
    (2, 1600, 100, 1296, "256x128"), (2, 4480, 91, 447, "256x128"), (2, 1280, 80, 1430, "256x128"), (1, 4096, 86, 457, "256x128"),      # 33.9 44.1, 31.2 42.1, 31.2 38.0, 30.7 40.5
    (2, 1024, 64, 1696, "128x128"), (2, 4096, 64, 512, "128x128"), (2, 640, 40, 1034, "128x128"), (2, 1600, 100, 250, "128x128")])       # one piece of either, short, and cut itself
def test_one_piece_of_a_long_k_on_128_x_128_tiles(launches, size, n, stages, columns, tiles):
    assert kernels_of(launches, size, n, columns, stages)[0] == "spmm_pipe " + tiles


@pytest.mark.parametrize("n,stages,columns", SLIM_TILES)
def test_products_tested_on_the_gpu_take_128_x_64_tiles_in_pieces_or_whole(launches, n, stages, columns):
    """In pieces from 29 stages on, but the tallest weights of the list."""
    for size in (1, 2):
        made = kernels_of(launches, size, n, columns, stages)
        assert made == ["spmm_pipe 128x64"] + ["spmm_reduce_splits 128x64"] * (stages >= 29 and n < 16384)


def test_pieces_fit_one_round_of_compute_units():
    """Read off the scratch that a product asks for, in partial tiles of the size that it takes: whole pieces, of no more tiles than there are units."""
    from sparse import _native as N
    for n, k, columns, rows in ((11008, 11008, 48, 128), (5120, 32768, 32, 128), (12288, 16384, 64, 128), (17408, 32768, 64, 256), (33024, 11008, 64, 256)):
        tile, tiles = rows * 64 * 4, -(-n // rows)
        blocks, rest = divmod(N.lib().tf24_spmm_workspace_bytes(N.E4M3, n, k, columns), tile)
        assert rest == 0 and blocks <= 256 and blocks % tiles == 0 and blocks != tiles, (n, k)
        assert (blocks > 0) == (n < 32768), (n, k)
