"""The rules by which a product chooses its tiles, called on the CPU as the launch code calls them."""
import ctypes
import importlib.util
import os
import subprocess

import pytest

from test_gpu_parity import LOWER_TILES, MID_TILES, NOT_TALL, SHORT, SLIM_TILES, SMALL_TILES, SQUARE, SQUARE_STRIDED, STAGE_ORDER, TALL
from test_gpu_training import MANY_LONG

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
extern "C" int small(int64_t n_sparse, int64_t n_dense, int stages, int bytes) {
  const int64_t ws = (int64_t)1 << 40;
  if (bytes == 1) return tf24::takes_small<tf24::e4m3_t>(n_sparse, (int64_t)stages * 128, n_dense, ws) * tf24::choose_pieces<tf24::e4m3_t, tf24::SmallCfg>(n_sparse, (int64_t)stages * 128, n_dense, ws, false).count;
  return tf24::takes_small<tf24::f16_t>(n_sparse, (int64_t)stages * 64, n_dense, ws) * tf24::choose_pieces<tf24::f16_t, tf24::SmallCfg>(n_sparse, (int64_t)stages * 64, n_dense, ws, false).count;
}
extern "C" int lower(int64_t n_sparse, int64_t n_dense, int stages, int bytes) {
  return bytes == 1 ? tf24::takes_lower<tf24::e4m3_t>(n_sparse, (int64_t)stages * 128, n_dense, (int64_t)1 << 40)
                    : tf24::takes_lower<tf24::f16_t>(n_sparse, (int64_t)stages * 64, n_dense, (int64_t)1 << 40);
}
extern "C" int mid(int64_t n_sparse, int64_t n_dense, int stages) {
  return tf24::takes_mid<tf24::f16_t>(n_sparse, (int64_t)stages * 64, n_dense, (int64_t)1 << 40);
}
extern "C" int64_t narrow(int64_t n_sparse, int64_t panels, int eight_bit) { return tf24::narrow_columns(n_sparse, panels, eight_bit); }
extern "C" int rotate_from() { return tf24::kRotateMinStages; }
""")
    subprocess.run([build.HIPCC, *build.FLAGS, "--offload-host-only", "-shared", str(src), "-o", str(lib)], check=True, capture_output=True)
    handle = ctypes.CDLL(str(lib))
    handle.square.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_int]
    handle.tiles.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_int]
    handle.tiles_of_16_bits.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_int]
    handle.strided.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int]
    handle.strided_pieces.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    handle.small.argtypes = handle.lower.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_int]
    handle.mid.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    handle.narrow.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    handle.narrow.restype = ctypes.c_int64
    return handle


@pytest.mark.parametrize("n,panels,columns,narrow", [
    # measured apart (us on the kernels for few columns, on 128 x 64 tiles)
    (5120, 20, 16, 1), (4096, 64, 24, 1), (4096, 28, 32, 1), (2304, 12, 40, 1), (4096, 172, 16, 1),     # 6.0 7.2, 8.6 9.5, 5.6 8.7, 4.9 5.7, 14.6 14.8
    (736, 80, 16, 0), (1600, 100, 24, 0), (6144, 64, 32, 0), (9824, 7, 32, 0), (4320, 19, 48, 0), (3840, 20, 64, 0)])    # 8.7 8.1, 10.9 8.9, 13.5 10.8, 6.0 5.0, 11.1 7.1, 9.1 7.4
def test_kernels_for_few_columns_where_they_are_the_faster_ones(rules, n, panels, columns, narrow):
    assert (columns <= rules.narrow(n, panels, 0)) == narrow


@pytest.mark.parametrize("n,stages,columns", SLIM_TILES + MID_TILES)
def test_products_tested_on_the_gpu_take_the_tiles_of_64_and_128_columns(rules, n, stages, columns):
    for size in (1, 2):
        if columns <= 64:
            assert columns > rules.narrow(n, stages, size == 1)
        else:
            assert rules.mid(n, columns, stages) and not rules.small(n, columns, stages, size) and not rules.lower(n, columns, stages, size)


@pytest.mark.parametrize("n,stages,columns,small", [
    # measured apart (us on the other tiles, on 128 x 128 ones)
    (768, 12, 160, 1), (3072, 12, 952, 1), (4096, 64, 128, 1), (6144, 64, 424, 1),              # 8.6 6.8, 9.2 7.6, 16.0 14.4, 28.9 21.5
    (5824, 159, 328, 0), (9024, 163, 272, 0), (2048, 320, 760, 0),                              # 47 63, 60 72, 57 81
    (5120, 20, 840, 0), (768, 12, 64, 0)])                                                      # two rounds of them; the narrowest tiles
def test_small_tiles_where_they_are_the_faster_ones(rules, n, stages, columns, small):
    assert bool(rules.small(n, columns, stages, 2)) == small


@pytest.mark.parametrize("n,stages,columns,lower", [
    # measured apart (us on 256 x 128 tiles, on 192 x 128 ones)
    (3840, 20, 1040, 1), (6144, 64, 736, 1), (11008, 64, 336, 1), (2048, 128, 2928, 1),         # 13.6 12.4, 34.1 30.1, 40.7 32.6, 79.7 65.7
    (2304, 12, 2368, 0), (5952, 189, 784, 0), (4096, 64, 512, 0), (4096, 64, 1536, 0)]          # 10.6 11.3, 95 100; 128 x 128; two rounds
    + [(*case, 1) for case in LOWER_TILES])
def test_lower_tiles_where_they_are_the_faster_ones(rules, n, stages, columns, lower):
    for size in (1, 2):
        assert rules.lower(n, columns, stages, size) == lower and not (lower and rules.small(n, columns, stages, size))


@pytest.mark.parametrize("n,stages,columns", SMALL_TILES)
def test_products_tested_on_the_gpu_take_small_tiles(rules, n, stages, columns):
    for size in (1, 2):
        assert bool(rules.small(n, columns, stages, size))
        assert stages <= 28 or rules.small(n, columns, stages, size) > 1


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


@pytest.mark.parametrize("n,stages,rows,form16,form8", SHORT)
def test_products_of_few_stages_tested_on_the_gpu_take_the_tiles_they_are_for(rules, n, stages, rows, form16, form8):
    codes = {"wide": 0, "narrow": 2, "square": 3, "tall": 4}
    assert (rules.tiles_of_16_bits(n, rows, stages, CU_SLOTS), rules.tiles(n, rows, stages, 1, CU_SLOTS)) == (codes[form16], codes[form8])
    assert rules.tiles(n, rows, stages, 0, CU_SLOTS) == 0                     # 32-bit results stay on 256 x 256 tiles
    assert -(-n // 256) * -(-rows // 128) > 256


@pytest.mark.parametrize("n,stages,columns,form", [
    # measured (us on the other tiles, on the form taken): rounds that other widths fill better, or do not
    (3072, 12, 12288, 2), (5120, 20, 4096, 2), (4800, 25, 4096, 2), (4096, 15, 4145, 4),              # 41.8 39.0, 40.0 36.2, 47.0 41.9, 26.1 23.3
    (4096, 16, 8192, 0), (6400, 25, 6144, 0), (5280, 12, 8114, 0),                                    # 40.5 46.3, 75.8 81.2, 46.8 53
    (2048, 8, 6144, 0), (2304, 12, 4096, 2)])                                                         # 13.1 13.6, 14.3 13.7
def test_tiles_of_products_of_few_stages(rules, n, stages, columns, form):
    assert rules.tiles_of_16_bits(n, columns, stages, CU_SLOTS) == form


@pytest.fixture(scope="module")
def dense_rules(tmp_path_factory):
    spec = importlib.util.spec_from_file_location("tf24_build", os.path.join(ROOT, "2by4-pretrain_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    folder = tmp_path_factory.mktemp("dense_rules")
    handles = []
    for source, rule in (
            ("dense_linear.hip", "linear(int64_t rows, int64_t k, int64_t tokens) { return tf24::shapes_fit(rows, k, tokens) && tf24::suits(rows, k, tokens, 256); }"),
            ("grad_weight.hip", "gradient(int64_t tokens, int64_t m, int64_t n) {\n"
                                "  const int64_t any = (int64_t)1 << 40;\n"
                                "  return !tf24::takes_square(tokens, m, n, any) ? 0 : tf24::takes_long(tokens, m, n, any) ? 2 : 1;\n}")):
        src, lib = folder / ("rules_" + source), folder / (source + ".so")
        # (the rules alone: no kernel is instantiated, and what the source shares with the rest of the library stays undefined)
        src.write_text('#include "lds_copies.hpp"\n#undef hipLaunchKernelGGL\n#define hipLaunchKernelGGL(...) (void)0\n'
                       f'#include "{source}"\nextern "C" int {rule}\n')
        subprocess.run([build.HIPCC, *build.FLAGS, "--offload-host-only", "-shared", "-Wl,--unresolved-symbols=ignore-all", str(src), "-o", str(lib)],
                       check=True, capture_output=True)
        handles.append(ctypes.CDLL(str(lib), mode=os.RTLD_LAZY))
    for handle, name in zip(handles, ("linear", "gradient")):
        getattr(handle, name).argtypes = [ctypes.c_int64] * 3
    return handles


@pytest.mark.parametrize("rows,k,tokens,taken", [
    # measured (us in the library, in the kernel): several rounds of tiles, filled to 0.89 and more or not
    (3072, 768, 12288, 1), (768, 3072, 12288, 1), (2560, 640, 13317, 1),             # 60.1 56.3, 59.7 48.0, 58.6 44.8
    (4096, 1024, 4053, 0), (6400, 1600, 2525, 0),                                    # 29.0 35.3, 40.2 51.9
    # one round of long tiles (0.72) and of short ones (0.55)
    (1600, 6400, 2831, 0), (640, 2560, 10655, 1), (5120, 1280, 1074, 1), (4096, 1024, 1256, 0),          # 62.5 77.5, 46.0 37.2, 22.9 20.2, 15.2 16.4
    # what the kernel does not take at all
    (3076, 768, 12288, 0), (3072, 800, 12288, 0), (3072, 192, 12288, 0), (3072, 768, 0, 0), (0, 768, 12288, 0)])
def test_dense_products_are_taken_where_the_kernel_is_the_faster_one(dense_rules, rows, k, tokens, taken):
    assert dense_rules[0].linear(rows, k, tokens) == taken


@pytest.mark.parametrize("tokens,m,n,form", [
    # measured (us on 32 x 32 instructions, on 16 x 16 ones): at least 160 blocks of at least 1024 tokens, or less
    (12288, 3072, 768, 2), (12288, 768, 3072, 2), (16384, 2048, 512, 2), (4423, 5120, 1280, 2),          # 65.2 62.5, 65.5 63.7, 48.9 47.5, 65.8 63.9
    (2000, 1024, 4096, 1), (745, 3072, 768, 1), (5000, 512, 2048, 1)]                                    # 32.8 33.7, 16.9 17.4, 24.6 25.2
    + [(*sizes, 2) for sizes in MANY_LONG])
def test_weight_gradients_take_long_tiles_where_they_are_the_faster_ones(dense_rules, tokens, m, n, form):
    assert dense_rules[1].gradient(tokens, m, n) == form
