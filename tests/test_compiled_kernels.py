"""Properties of the tiled 2:4 kernels that a result cannot show, read from the assembly that hipcc makes of this
repository's sources: whether the copies of a stage may stay in flight over the stage barrier, and what is spilled."""
import importlib.util
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _assembly(tmp_path, kernels):
    """{kernel symbol: its lines} of spmm_pipe instantiated for each of `kernels` (template arguments)"""
    spec = importlib.util.spec_from_file_location("tf24_build", os.path.join(ROOT, "2by4-pretrain_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    src, out = tmp_path / "kernels.hip", tmp_path / "kernels.s"
    src.write_text('#include "spmm_kernels.hpp"\nnamespace tf24 { const void* kernels[] = {'
                   + ", ".join(f"(const void*)spmm_pipe<{k}>" for k in kernels) + "}; }\n")
    subprocess.run([build.HIPCC, *build.FLAGS, "--cuda-device-only", "-S", str(src), "-o", str(out)], check=True, capture_output=True)
    found, lines = {}, None
    for line in out.read_text().splitlines():
        start = re.match(r"(_Z\w*spmm_pipe\w*):\s*; @", line)
        if start:
            lines = found[start.group(1)] = []
        elif line.startswith(".Lfunc_end"):
            lines = None
        elif lines is not None:
            lines.append(line)
    assert len(found) == len(kernels)
    return found


def _stage_loop(lines):
    """The first innermost loop with matrix instructions."""
    labels, loops = {}, []
    for i, line in enumerate(lines):
        label = re.match(r"(\.LBB\w+):", line)
        if label:
            labels[label.group(1)] = i
        branch = re.search(r"s_c?branch\w*\s+(\.LBB\w+)", line)
        if branch and branch.group(1) in labels:
            loops.append((labels[branch.group(1)], i))
    loops = [(a, b) for a, b in loops if any("smfmac" in line for line in lines[a:b])]
    a, b = min((a, b) for a, b in loops if not any((c, d) != (a, b) and a <= c and d <= b for c, d in loops))
    return lines[a:b]


def test_chained_tiles_wait_only_at_the_stage_barrier(tmp_path):
    """The loop over the stages waits for memory once, at its barrier, with the next stage's copies left in flight."""
    kernels = [f"{t}, {out}, true, {tile}, {strided}, true, {acts}"
               for t, out, tile, strided, acts in (
                   ("f16_t", "f16_t", "TiledCfg", "false", "false"), ("f16_t", "f16_t", "TiledCfg", "true", "false"),
                   ("bf16_t", "bf16_t", "TiledCfg", "false", "false"), ("f16_t", "float", "TiledCfg", "false", "false"),
                   ("f16_t", "float", "TiledCfg", "true", "true"), ("f16_t", "f16_t", "SquareCfg", "false", "false"),
                   ("f16_t", "f16_t", "Wave4Cfg", "false", "false"), ("f16_t", "f16_t", "Wave4Cfg192", "false", "false"),
                   ("f16_t", "f16_t", "TallCfg", "false", "false"), ("bf16_t", "bf16_t", "TallCfg", "false", "true"))]
    for name, lines in _assembly(tmp_path, kernels).items():
        waits = [int(n) for line in _stage_loop(lines) for n in re.findall(r"vmcnt\((\d+)\)", line)]
        assert len(waits) == 1 and waits[0] > 0, (name, waits)


def test_activation_forms_spill_nothing(tmp_path):
    """The 8-wave kernels with an activation, the ones nearest to their 256 registers, keep everything in them."""
    kernels = [f"{t}, {out}, true, TiledCfg, {strided}, {chained}, true"
               for t, out, strided, chained in (
                   ("f16_t", "f16_t", "false", "true"), ("f16_t", "f16_t", "true", "true"), ("f16_t", "f16_t", "true", "false"),
                   ("bf16_t", "bf16_t", "false", "true"), ("e4m3_t", "bf16_t", "false", "true"), ("e4m3_t", "f16_t", "false", "true"))]
    for name, lines in _assembly(tmp_path, kernels).items():
        assert not any("scratch_" in line for line in lines), name


def test_four_wave_forms_spill_outside_the_stage_loop_only(tmp_path):
    """Tiles of the 4-wave forms keep every vector register, and what they put aside of the scalar ones stays aside while stages are multiplied."""
    kernels = [f"f16_t, f16_t, true, {tile}, false, true, {acts}" for tile in ("TallCfg", "Wave4Cfg", "Wave4Cfg192", "SquareCfg") for acts in ("false", "true")]
    for name, lines in _assembly(tmp_path, kernels).items():
        assert not any("scratch_" in line for line in lines), name
        assert not any("v_writelane" in line or "v_readlane" in line for line in _stage_loop(lines)), name


def test_compression_by_magnitude_streams_its_loads_only(tmp_path):
    """What it reads leaves the caches to what it wrote, which is used next: streaming loads, ordinary stores."""
    spec = importlib.util.spec_from_file_location("tf24_build", os.path.join(ROOT, "2by4-pretrain_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    out = tmp_path / "prune_compress.s"
    subprocess.run([build.HIPCC, *build.FLAGS, "--cuda-device-only", "-S", os.path.join(build.CSRC, "prune_compress.hip"), "-o", str(out)],
                   check=True, capture_output=True)
    text = out.read_text()
    for kernel in ("prune_compress_row_mag16_panelINS_6bf16_tENS_5f16_tE", "prune_compress_rowIfNS_5f16_tELi0EhLb1E"):
        (body,) = re.findall(rf"^_Z\w*{kernel}\w*:.*?^\.Lfunc_end", text, flags=re.S | re.M)
        loads, stores = re.findall(r"global_load_dwordx4.*", body), re.findall(r"global_store_dwordx2.*", body)
        assert loads and all(line.endswith(" nt") for line in loads), (kernel, loads)
        assert stores and not any(line.endswith(" nt") for line in stores), (kernel, stores)


@pytest.mark.parametrize("columns,waves", [(8, 2), (16, 4), (32, 8)])
def test_lanes_that_exchange_data_through_lds_are_ordered(tmp_path, columns, waves):
    """What a wave of the kernel for few columns writes to its slice of LDS and what other lanes read there are ordered by a fence, either way
    round, in the code as it is optimised."""
    spec = importlib.util.spec_from_file_location("tf24_build", os.path.join(ROOT, "2by4-pretrain_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    src, out = tmp_path / "few.hip", tmp_path / "few.ll"
    src.write_text(f"""#include "spmm_kernels.hpp"
void few() {{
  hipLaunchKernelGGL((tf24::spmm_few<tf24::f16_t, tf24::f16_t, true, {columns}, {waves}>), dim3(1), dim3({64 * waves}), 0, 0, nullptr, nullptr, 16, 64, nullptr, 64, 1,
                     nullptr, 16, nullptr, 1.0f, 0);
}}
""")
    subprocess.run([build.HIPCC, *build.FLAGS, "--offload-device-only", "-S", "-emit-llvm", str(src), "-o", str(out)], check=True, capture_output=True)
    last, fenced, changes = None, True, 0
    for line in out.read_text().splitlines():
        if "fence syncscope(\"wavefront\")" in line:
            fenced = True
        elif "addrspace(3)" in line and ("store <4 x i32>" in line or "load <4 x i32>" in line):       # (the partial sums are floats)
            access = "store" if "store <4 x i32>" in line else "load"
            if last not in (None, access):
                assert fenced, line
                changes += 1
            last, fenced = access, False
    assert changes >= 3


def test_dense_products_and_conversions_order_the_lanes_that_exchange_data_through_lds(tmp_path):
    """The staged results of the dense product's output pass, and what the panel conversion exchanges: between writes to LDS and reads of it, either way
    round, stands a fence or a barrier's clobber in the code as it is optimised."""
    spec = importlib.util.spec_from_file_location("tf24_build", os.path.join(ROOT, "2by4-pretrain_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    for source, wanted in (("dense_linear.hip", "dense_linear"), ("prune_compress.hip", "mag16_panel")):
        out = tmp_path / "out.ll"
        subprocess.run([build.HIPCC, *build.FLAGS, "--offload-device-only", "-S", "-emit-llvm", os.path.join(build.CSRC, source), "-o", str(out)], check=True, capture_output=True)
        found, inside = 0, False
        for line in out.read_text().splitlines():
            label = re.match(r"(\d+):.*; preds = (.*)", line)
            if line.startswith("define "):
                inside, last, ordered, changes, block = wanted in line, None, True, 0, None
            elif label:
                if block is not None and f"%{block}" not in label.group(2).split(", "):
                    last, ordered = None, True                               # not entered from the block above it
                block = label.group(1)
            elif line == "}" and inside:
                found, inside = found + (changes > 0), False
            elif inside and (line.lstrip().startswith("fence ") or "~{memory}" in line):
                ordered = True
            elif inside and "addrspace(3)" in line and (" store " in line or re.search(r" load (<\d x i\d+>|i64|i32)", line)):      # (pieces as they are stored; not the bias)
                access = "store" if " store " in line else "load"
                if last not in (None, access):
                    assert ordered, (wanted, line)
                    changes += 1
                last, ordered = access, False
        assert found >= 3, wanted
