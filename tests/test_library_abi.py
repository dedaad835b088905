"""CPU-side checks of the C-ABI library and the Python boundary: the library loads without a
GPU, exports every symbol include/tf24.h declares, its host-only validators reproduce the
reference's argument errors, and the Python API fails loudly instead of falling back."""
import ctypes
import importlib.util
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "tf24.h")


@pytest.fixture(scope="module")
def native():
    from sparse import _native
    if not os.path.exists(_native.library_path()):      # build only when nothing is built
        spec = importlib.util.spec_from_file_location("tf24_build", os.path.join(ROOT, "2by4-pretrain_amd", "build.py"))
        mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
        mod.build_library()
    return _native


def _declared_symbols():
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    return sorted(set(re.findall(r"\b(tf24_[a-z0-9_]+)\s*\(", text)))


def test_header_symbols_are_exported(native):
    names = _declared_symbols()
    assert len(names) >= 13 and "tf24_spmm" in names and "tf24_prune_compress" in names
    handle = ctypes.CDLL(native.library_path())
    for name in names:
        assert hasattr(handle, name), f"{name} declared in tf24.h but not exported"
    # and the binding knows every declared entry point
    assert set(names) == set(native._SIGNATURES)


def test_version_and_error_string(native):
    assert native.version().startswith("tf24 ") and "gfx950" in native.version()
    lib = native.lib()
    rc = lib.tf24_prune_compress_validate(native.F16, native.ROW_MAJOR, 64, 33, 64, native.PRUNE_MAGNITUDE, 0, 0, 0, 0, 0, native.F16)
    assert rc == -1 and b"multiple of (32, 64)" in lib.tf24_last_error()


@pytest.mark.parametrize("m,k,out,ok", [(32, 64, 1, True), (32, 128, 3, True), (32, 64, 3, False), (48, 64, 1, False),
                                        (32, 96, 1, False), (16, 64, 1, False), (3072, 768, 1, True), (11008, 4096, 2, True)])
def test_compress_shape_rules(native, m, k, out, ok):
    # sparse/semi_structured.py:24-30,188-200: rows % 32, cols % 64 (16-bit) / 128 (8-bit), and at least that
    rc = native.lib().tf24_prune_compress_validate(native.F32, native.ROW_MAJOR, k, m, k, native.PRUNE_MAGNITUDE, 0, 0, 0, 0, 0, out)
    assert (rc == 0) == ok


def test_compress_argument_rules(native):
    lib, N = native.lib(), native
    ok = dict(in_dtype=N.BF16, layout=N.ROW_MAJOR, ld=64, m=32, k=64, mode=N.PRUNE_MAGNITUDE, has_mask=0, mask_dtype=N.U8, mask_ld=0,
              has_rand=0, rand_ld=0, out=N.F16)

    def call(**kw):
        a = dict(ok, **kw)
        return lib.tf24_prune_compress_validate(a["in_dtype"], a["layout"], a["ld"], a["m"], a["k"], a["mode"], a["has_mask"],
                                                a["mask_dtype"], a["mask_ld"], a["has_rand"], a["rand_ld"], a["out"])
    assert call() == 0
    assert call(in_dtype=N.E4M3) == -2 and call(out=N.F32) == -2 and call(out=N.U8) == -2
    assert call(layout=7) == -5 and call(mode=9) == -5
    assert call(ld=32) == -3 and call(ld=68) == -3                      # too small / not a multiple of 8
    assert call(layout=N.COL_MAJOR, ld=32) == 0 and call(layout=N.COL_MAJOR, ld=24) == -3
    assert call(mode=N.PRUNE_MASK) == -5                                 # mask missing
    assert call(mode=N.PRUNE_MASK, has_mask=1, mask_ld=64) == 0
    assert call(mode=N.PRUNE_MASK, has_mask=1, mask_ld=64, mask_dtype=N.E4M3) == -2
    assert call(mode=N.PRUNE_MVUE) == -5                                 # uniforms missing
    assert call(mode=N.PRUNE_MVUE, has_rand=1, rand_ld=64) == 0
    assert call(mode=N.PRUNE_MVUE, has_rand=1, rand_ld=64, has_mask=1, mask_ld=64) == -5   # MVUE with mask
    assert b"MVUE24 with mask" in lib.tf24_last_error()


def test_transposable_and_spmm_validators(native):
    lib, N = native.lib(), native
    assert lib.tf24_transposable_mask_validate(N.BF16, N.ROW_MAJOR, 64, 32, 64) == 0
    assert lib.tf24_transposable_mask_validate(N.BF16, N.ROW_MAJOR, 64, 33, 64) == -1       # transposable_semi_structured.py:60-63
    assert lib.tf24_transposable_mask_validate(N.BF16, N.ROW_MAJOR, 32, 32, 32) == -1       # :64-67
    assert lib.tf24_transposable_mask_validate(N.E4M3, N.ROW_MAJOR, 64, 32, 64) == -2       # :58-59
    assert lib.tf24_transposable_mask_validate(N.F32, N.COL_MAJOR, 32, 32, 64) == 0
    # csrc .cu:101-109: sparse rows % 32, k % 64 | 128, dense extent % 8 | 16
    sp = lambda dt, n, k, nd, **kw: lib.tf24_spmm_validate(dt, n, k, kw.get("bl", N.ROW_MAJOR), kw.get("ldb", k), nd,
                                                             kw.get("out", N.F16), kw.get("cl", N.COL_MAJOR), kw.get("ldc", n), kw.get("act", 0))
    assert sp(N.F16, 32, 64, 8) == 0 and sp(N.BF16, 11008, 4096, 8192) == 0 and sp(N.E4M3, 8192, 8192, 16384, out=N.BF16) == 0
    assert sp(N.F16, 48, 64, 8) == -1 and sp(N.F16, 32, 96, 8) == -1 and sp(N.F16, 32, 64, 12) == -1
    assert sp(N.E4M3, 32, 64, 16) == -1 and sp(N.E4M3, 32, 128, 8) == -1
    assert sp(N.F32, 32, 64, 8) == -2 and sp(N.F16, 32, 64, 8, out=N.E4M3) == -2
    assert sp(N.F16, 32, 64, 8, ldb=32) == -3 and sp(N.F16, 32, 64, 8, ldc=16) == -3
    # output rows leave as 16-byte segments: ldc % 8 for 16-bit results, % 4 for 32-bit ones
    assert sp(N.F16, 32, 64, 8, ldc=36) == -3 and sp(N.F16, 32, 64, 8, ldc=40) == 0 and sp(N.F16, 32, 64, 8, ldc=36, out=N.F32) == 0
    assert sp(N.F16, 32, 64, 8, ldb=1 << 23) == 0 and sp(N.F16, 32, 64, 8, ldb=(1 << 23) + 8) == -3     # rows of the dense operand: at most 16 MiB
    assert sp(N.E4M3, 32, 128, 16, ldb=1 << 24) == 0 and sp(N.E4M3, 32, 128, 16, ldb=(1 << 24) + 16) == -3
    assert sp(N.F16, 32, 64, 8, act=5) == -5 and sp(N.F16, 32, 64, 8, bl=3) == -5
    # a float32 bias, whatever the results are but integers
    assert sp(N.F16, 32, 64, 8, act=N.BIAS_F32) == 0 and sp(N.E4M3, 32, 128, 16, out=N.F32, act=N.BIAS_F32 | N.ACT_GELU) == 0
    assert sp(N.F16, 32, 64, 8, act=N.BIAS_F32 | 5) == -5 and sp(N.I8, 32, 128, 16, out=N.I32, act=N.BIAS_F32) == -5


def test_misaligned_pointers_are_refused_before_any_launch(native):
    """The kernels use 128-bit accesses: entry points return TF24_ERR_STRIDE for a misaligned
    pointer instead of launching (no GPU is touched on this path, the addresses are made up)."""
    lib, N = native.lib(), native
    ok, off = 0x7f0000001000, 0x7f0000001008
    spmm = lambda a=ok, b=ok, c=ok, meta=ok: lib.tf24_spmm(a, meta, N.COMPRESSED_PANEL, N.F16, 64, 64, b, N.ROW_MAJOR, 64, 64,
                                                           c, N.F16, N.COL_MAJOR, 64, None, 1.0, 0, None, 0, None)
    assert spmm(b=off) == -3 and spmm(a=off) == -3 and spmm(c=off) == -3 and spmm(meta=ok + 4) == -3
    assert b"aligned" in lib.tf24_last_error()
    pc = lambda dense=ok, values=ok: lib.tf24_prune_compress(dense, N.F16, N.ROW_MAJOR, 64, 32, 64, N.PRUNE_MAGNITUDE, None, N.U8, 0,
                                                             None, 0, values, N.F16, ok, N.COMPRESSED_PANEL, None)
    assert pc(dense=off) == -3 and pc(values=off) == -3
    assert lib.tf24_transposable_mask(off, N.F16, N.ROW_MAJOR, 64, 32, 64, 1, None, ok, None) == -3
    assert lib.tf24_soft_threshold24(ok, N.F16, N.ROW_MAJOR, 64, 32, 64, off, ok, None) == -3
    assert lib.tf24_transpose(ok, N.F16, 64, 64, 64, off, 64, None) == -3
    assert lib.tf24_decompress(off, N.F16, ok, N.COMPRESSED_CANONICAL, 32, 64, ok, None) == -3


def test_int8_validators(native):
    """int8 values come from int8 matrices, take byte masks and no MVUE; the integer product gives
    int32 with no activation or ReLU (.cu:594-637)."""
    lib, N = native.lib(), native
    pc = lambda **a: lib.tf24_prune_compress_validate(a.get("dt", N.I8), a.get("layout", N.ROW_MAJOR), a.get("ld", 128), 32, 128,
                                                      a.get("mode", N.PRUNE_MAGNITUDE), a.get("has_mask", 0), a.get("mdt", N.U8),
                                                      a.get("mld", 0), a.get("has_rand", 0), a.get("rld", 0), a.get("out", N.I8))
    assert pc() == 0 and pc(mode=N.PRUNE_MASK, has_mask=1, mld=128) == 0
    assert pc(out=N.F16) == -2 and pc(dt=N.F16) == -2                    # int8 <-> int8 only
    assert pc(mode=N.PRUNE_MASK, has_mask=1, mld=128, mdt=N.F32) == -2   # byte masks only
    assert pc(mode=N.PRUNE_MVUE, has_rand=1, rld=128) == -5
    assert pc(layout=N.COL_MAJOR, ld=40) == -3 and pc(layout=N.COL_MAJOR, ld=48) == 0
    sp = lambda **a: lib.tf24_spmm_validate(N.I8, 32, 128, N.ROW_MAJOR, 128, 16, a.get("out", N.I32), N.COL_MAJOR, 32, a.get("act", 0))
    assert sp() == 0 and sp(act=N.ACT_RELU) == 0
    assert sp(out=N.F32) == -2 and sp(act=N.ACT_SILU) == -5 and sp(act=N.ACT_GELU) == -5
    assert lib.tf24_spmm_validate(N.F16, 32, 64, N.ROW_MAJOR, 64, 8, N.I32, N.COL_MAJOR, 32, 0) == -2
    assert lib.tf24_prune_compress_dual_validate(N.I8, 128, 128, 128, N.U8, 128, N.I8, N.COMPRESSED_PANEL) == 0
    assert lib.tf24_prune_compress_dual_validate(N.I8, 128, 128, 128, N.U8, 128, N.E4M3, N.COMPRESSED_PANEL) == -2
    assert lib.tf24_prune_compress_dual_validate(N.I8, 64, 64, 64, N.U8, 64, N.I8, N.COMPRESSED_PANEL) == -1


def test_dual_compress_validator(native):
    """Both W [m,k] and W^T [k,m] must be compressible: m and k multiples of 64 (128 for 8-bit values)."""
    lib, N = native.lib(), native
    dual = lambda m, k, **kw: lib.tf24_prune_compress_dual_validate(
        kw.get("dt", N.F32), kw.get("ld", k), m, k, kw.get("mdt", N.U8), kw.get("mld", k), kw.get("out", N.F16),
        kw.get("lay", N.COMPRESSED_PANEL))
    assert dual(64, 64) == 0 and dual(3072, 768) == 0 and dual(768, 3072, out=N.BF16, lay=N.COMPRESSED_CANONICAL) == 0
    assert dual(128, 256, out=N.E4M3) == 0 and dual(128, 256, out=N.E5M2, mdt=N.F32) == 0
    assert dual(96, 128) == -1 and dual(128, 96) == -1 and dual(32, 64) == -1
    assert dual(64, 128, out=N.E4M3) == -1 and dual(128, 192, out=N.E4M3) == -1
    assert dual(64, 64, dt=N.U8) == -2 and dual(64, 64, out=N.F32) == -2 and dual(64, 64, mdt=N.E4M3) == -2
    assert dual(64, 64, ld=56) == -3 and dual(64, 64, mld=68) == -3
    assert dual(64, 64, lay=2) == -5
    assert b"tf24_prune_compress_dual" in lib.tf24_last_error()


def test_python_api_rejects_cpu_tensors(native):
    import sparse
    with pytest.raises(RuntimeError, match="Only CUDA tensors"):
        sparse.to_sparse_semi_structured(torch.zeros(32, 64, dtype=torch.float16))
    with pytest.raises(RuntimeError):
        sparse.TransposableSparse()(torch.zeros(32, 64))
    with pytest.raises(RuntimeError):
        sparse.soft_threshold24_triton(torch.zeros(32, 64))
    with pytest.raises(AssertionError):
        sparse.masked_add_(torch.zeros(4), torch.zeros(4), torch.zeros(4), alpha=0.1)
    with pytest.raises(ValueError):
        sparse.SparseSemiStructuredTensor(None)


def test_missing_library_fails_loudly(native, monkeypatch):
    monkeypatch.setattr(native, "_lib", None)
    monkeypatch.setattr(native, "library_path", lambda: "/nonexistent/lib2by4_gfx950.so")
    with pytest.raises(RuntimeError, match="no fallback"):
        native.lib()


def test_product_path_does_not_import_the_oracle():
    pkg = os.path.join(ROOT, "2by4-pretrain_amd")
    for base, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".hpp", ".h")):
                text = open(os.path.join(base, f)).read()
                assert "import oracle" not in text and "from oracle" not in text, f


def test_reference_api_names_present():
    import sparse
    for name in ["to_sparse_semi_structured", "SparseSemiStructuredTensor", "TransposableSparse", "masked_add_",
                 "soft_threshold24_triton", "sparse24_triton", "MVUE24_approx_triton", "SparseLinearTranspose",
                 "sparse_linear_transpose"]:
        assert hasattr(sparse, name), name
    import inspect
    sig = inspect.signature(sparse.to_sparse_semi_structured)
    assert list(sig.parameters)[:5] == ["original_tensor", "transposed", "MVUE24", "mask", "dtype"]
    assert sig.parameters["dtype"].default is torch.float16
    cls = sparse.SparseSemiStructuredTensor
    assert cls._FORCE_CUTLASS is True and cls._FUSE_TRANSPOSE is False


def test_parameters_that_overlap_take_turns():
    """The optimizer updates the tensors of a round side by side: none of them may share memory, wherever they start, and of
    two that overlap the earlier one of the list goes first."""
    from sparse.adamw import _rounds
    base, other, empty = torch.zeros(100), torch.zeros(40), torch.zeros(0)

    def check(params, expected):
        rounds = _rounds(params)
        assert [[next(i for i, q in enumerate(params) if q is p) for p in r] for r in rounds] == expected

    check([base[:50], other, base[50:]], [[0, 1, 2]])
    check([base, base[4:], other], [[0, 2], [1]])
    check([base[4:], other, base], [[0, 1], [2]])
    check([base[:60], base[40:], base[:40]], [[0], [1, 2]])
    check([base, base[4:], base.view(10, 10), empty, torch.zeros(0)], [[0, 3, 4], [1], [2]])
    check([base[:1], base, base[99:]], [[0], [1], [2]])
    check([base.view(10, 10).t(), other.view(8, 5)], [[0, 1]])
    assert not any(_rounds([]))


def test_pieces_of_products_with_few_columns():
    """Pieces of k, read off the scratch that a product asks for (float32 partial tiles, 256 x 64 or two of 128 x 64, k-strided 256 x 256): their
    blocks fit one round of 256 compute units, partial tiles count for the columns that the dense operand
    reaches, and one pass over the weight asks for none."""
    from sparse import _native as N
    scratch = N.lib().tf24_spmm_workspace_bytes
    for code, n, k, columns in ((N.E4M3, 11008, 11008, 48), (N.E4M3, 5120, 32768, 32), (N.E4M3, 20480, 8192, 64), (N.F16, 12288, 8192, 64)):
        tile = 256 * (64 if code == N.E4M3 else 256) * 4                       # (16-bit types: k-strided, the larger tile)
        blocks = scratch(code, n, k, columns) // tile
        assert 0 < blocks <= 256 and blocks % ((n + 255) // 256) == 0, (n, k)
    for n, k in ((6144, 1536), (5120, 1024), (11008, 2048)):
        assert scratch(N.F16, n, k, 16) > 0
    for n, k in ((11008, 4096), (3072, 768), (8192, 8192)):
        assert scratch(N.F16, n, k, 1) == scratch(N.E4M3, n, k, 1) == scratch(N.E4M3, n, k, 8) == 0


def test_weights_saved_without_their_dtype_attribute(tmp_path):
    """A compressed weight that was saved before its objects carried the dtype loads and answers as a new one does."""
    from sparse import SparseSemiStructuredTensor
    new = SparseSemiStructuredTensor(None, torch.Size((32, 64)), sparse_tensor_cutlass=torch.ones(32, 32).half(),
                                     meta_tensor_cutlass=torch.zeros(32, 4, dtype=torch.int16))
    old = new.detach()
    del old.__dict__["_dtype"]
    for i, weight in enumerate((new, old)):
        torch.save(weight, tmp_path / f"{i}.pt")
        loaded = torch.load(tmp_path / f"{i}.pt", weights_only=False)
        for w in (loaded, loaded.detach(), loaded.t()):
            assert w._dtype is w.dtype is torch.float16 and w._out_dtype() is None


def test_other_tensor_classes_meet_a_compressed_weight(monkeypatch):
    """A 2:4 weight takes no part in what other classes do with torch's functions: a plain subclass of Tensor keeps its class, one
    whose handler declines classes that it does not know is asked without this one, as beside a dense weight."""
    import torch.nn.functional as F
    from sparse import SparseSemiStructuredTensor, semi_structured
    monkeypatch.setattr(semi_structured, "_spmm", lambda s, x, first, **kw: torch.full((x.shape[0], 32), 2.0, dtype=x.dtype))
    weight = SparseSemiStructuredTensor(None, torch.Size((32, 64)), sparse_tensor_cutlass=torch.ones(32, 32).half(),
                                        meta_tensor_cutlass=torch.zeros(32, 4, dtype=torch.int16))

    class Plain(torch.Tensor):
        pass

    class Handler(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            return types if all(issubclass(t, Handler) for t in types) else NotImplemented

    class Declines(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            return NotImplemented

    x = torch.ones(8, 64).half()
    for grad in (False, True):
        with torch.set_grad_enabled(grad):
            for call in (lambda x: F.linear(x, weight), lambda x: torch.mm(x, weight.t())):
                for cls in (torch.Tensor, Plain):
                    out = call(x.as_subclass(cls))
                    assert type(out) is cls and out.shape == (8, 32)
                assert call(x.as_subclass(Handler)) == (Handler,)
                with pytest.raises(TypeError):
                    call(x.as_subclass(Declines))
            assert torch.mm(weight, x.t().as_subclass(Handler)) == (Handler,)
            assert F.linear(x, weight, torch.ones(32).as_subclass(Handler)) == (Handler,)


def test_derived_weights_handle_their_own_methods():
    """A class derived from the 2:4 weights with a __torch_function__ of its own sees t, values and indices; one without has the
    weight's."""
    from sparse import SparseSemiStructuredTensor

    class Derived(SparseSemiStructuredTensor):
        pass

    class Handles(SparseSemiStructuredTensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            return func.__name__

    make = lambda cls: cls(None, torch.Size((32, 64)), sparse_tensor_cutlass=torch.ones(32, 32).half(),
                           meta_tensor_cutlass=torch.zeros(32, 4, dtype=torch.int16))
    handles = make(Handles)
    assert (handles.t(), handles.values(), handles.indices()) == ("t", "values", "indices")
    for cls in (Derived, SparseSemiStructuredTensor):
        weight = make(cls)
        assert weight.t().shape == (64, 32) and weight.t().transposed
        assert weight.values().shape == (32, 32) and weight.indices().shape == (32, 4)


def test_fast_calls_take_what_ctypes_takes():
    """The CPython module's functions over the same library: the same results and the same refusals as through ctypes."""
    import ctypes

    import pytest
    from sparse import _fastcall, _native as N
    fast = N.lib()
    slow = ctypes.CDLL(N.library_path())
    names = [n for n in N._SIGNATURES if hasattr(_fastcall, n)]
    assert "tf24_spmm" in names and "tf24_linear" in names and all(getattr(fast, n) is getattr(_fastcall, n) for n in names)
    for name in names:
        res, types = N._SIGNATURES[name]
        fn = getattr(slow, name)
        fn.restype, fn.argtypes = res, types
        # null pointers and empty shapes: every entry point answers these on the host
        args = [None if t is ctypes.c_void_p else 0 if t in (ctypes.c_int, ctypes.c_int64) else 0.0 for t in types]
        assert getattr(fast, name)(*args) == fn(*args), name
        for bad in (args[:-1], [*args[:-1], "x"], [1.5 if t in (ctypes.c_int, ctypes.c_int64) else a for t, a in zip(types, args)] if ctypes.c_int64 in types else args[:-1]):
            with pytest.raises(TypeError):
                getattr(fast, name)(*bad)
    for shape in ((3072, 768, 12288), (4096, 11008, 37), (8, 64, 1), (True, 64, 64)):
        for code in (N.F16, N.E4M3, N.I8):
            assert fast.tf24_spmm_workspace_bytes(code, *shape) == slow.tf24_spmm_workspace_bytes(code, *shape)
    assert fast.tf24_linear16_suits(2 ** 64 + 3072, 768, 12288) == slow.tf24_linear16_suits(2 ** 64 + 3072, 768, 12288) == 1      # modulo 2^64, as ctypes does
    assert fast.tf24_adamw_masked_decay_list(b"", 0, 0, 0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0, None) == slow.tf24_adamw_masked_decay_list(b"", 0, 0, 0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0, None)


def test_fast_calls_take_numbers_and_objects_of_ctypes():
    """Floating-point arguments arrive as they are (the refusal of hyper-parameters names them), and what ctypes takes besides plain numbers is taken."""
    from sparse import _native as N
    fast = N.lib()
    slow = ctypes.CDLL(N.library_path())
    slow.tf24_last_error.restype = ctypes.c_char_p
    slow.tf24_adamw_masked_decay_list.argtypes = N._SIGNATURES["tf24_adamw_masked_decay_list"][1]
    slow.tf24_decompress.argtypes = N._SIGNATURES["tf24_decompress"][1]
    outcomes = []
    for numbers in ((1e-3, 1.25, 0.999, 1e-8, 0.0, 0.0), (2, -0.5, 0.875, 3e-7, 1, 0), tuple(map(ctypes.c_double, (1e-3, 1.25, 0.999, 1e-8, 0.0, 0.0)))):
        for lib in (fast, slow):
            assert lib.tf24_adamw_masked_decay_list(None, 0, 0, 0, *numbers, 1, None) != 0
            outcomes.append(lib.tf24_last_error())
        assert outcomes[-1] == outcomes[-2]
    assert outcomes[0] == outcomes[4] and b"lr 0.001, eps 1e-08, betas 1.25 0.999" in outcomes[0] and b"lr 2, eps 3e-07, betas -0.5 0.875" in outcomes[2]
    # pointers: a misaligned one is refused before anything is read from it
    buffer = (ctypes.c_char * 80)()
    at = ctypes.addressof(buffer) | 1
    odd = (ctypes.c_char * 8).from_address(at)
    for lib in (fast, slow):
        for values in (at, ctypes.c_void_p(at), odd, ctypes.byref(odd), ctypes.pointer(odd)):
            assert lib.tf24_decompress(values, N.F16, ctypes.c_void_p(64), ctypes.c_int(0), ctypes.c_int64(32), 64, 64, None) != 0
            assert b"aligned" in lib.tf24_last_error(), lib.tf24_last_error()
        with pytest.raises((TypeError, ctypes.ArgumentError)):
            lib.tf24_decompress(1.5, N.F16, 64, 0, 32, 64, 64, None)


@pytest.mark.parametrize("missing", [True, False])
def test_library_loads_without_the_cpython_module(missing, monkeypatch):
    """Not built, or built for another interpreter: ctypes makes the calls.  Only a missing library is an error, and says how to build it."""
    import sys

    import sparse
    from sparse import _native as N
    N.lib()
    monkeypatch.setattr(N, "_lib", None)
    monkeypatch.delattr(sparse, "_fastcall", raising=False)
    if missing:
        monkeypatch.setitem(sys.modules, "sparse._fastcall", None)           # (its import raises ImportError)
        lib = N.lib()
        assert isinstance(lib.tf24_spmm, ctypes._CFuncPtr) and lib.tf24_linear16_suits(3072, 768, 12288) == 1
    else:
        monkeypatch.setattr(N, "library_path", lambda: os.path.join(ROOT, "nowhere", "lib2by4_gfx950.so"))
        with pytest.raises(RuntimeError, match="build.py"):
            N.lib()


def test_cpython_module_says_which_interpreters_it_fits():
    import importlib.machinery

    from sparse import _fastcall
    suffix = os.path.basename(_fastcall.__file__)[len("_fastcall"):]
    assert suffix == ".abi3.so" and suffix in importlib.machinery.EXTENSION_SUFFIXES
