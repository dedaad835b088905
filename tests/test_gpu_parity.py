"""GPU parity: every HIP kernel, called through the Python API -> ctypes -> C ABI, against the CPU
oracle on the same seeded inputs.  Bit-exact for masks, metadata, compressed values and the
element-wise operators; stated tolerances for the matmul."""
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

F16, BF16, F32, E4M3, E5M2 = torch.float16, torch.bfloat16, torch.float32, torch.float8_e4m3fn, torch.float8_e5m2
FLOAT8 = (E4M3, E5M2)


def bits(t):
    t = t.detach().cpu().contiguous()
    if t.dtype == torch.bool:
        return t
    return t.view({1: torch.uint8, 2: torch.int16, 4: torch.int32}[t.element_size()])


def assert_same(got, want, what=""):
    assert got.shape == want.shape, (what, got.shape, want.shape)
    assert got.dtype == want.dtype, (what, got.dtype, want.dtype)
    g, w = bits(got), bits(want)
    if not g.equal(w):
        bad = (g != w).nonzero()
        raise AssertionError(f"{what}: {bad.shape[0]} of {g.numel()} elements differ, first at {bad[0].tolist()}: "
                             f"got {got.detach().cpu()[tuple(bad[0])]} want {want[tuple(bad[0])]}")


def randn(shape, dtype, seed, scale=1.0, ties=False):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(shape, generator=g) * scale
    if ties:   # coarse grid: many equal magnitudes inside groups
        x = torch.round(x * 2) / 2
    return x.to(dtype)


def maybe_t(x, col_major):
    """A logical tensor equal to x, stored column-major when asked (like W.T of a row-major W)."""
    return x.t().contiguous().t() if col_major else x


# ------------------------------------------------------------------ prune + compress
@pytest.mark.parametrize("col_major", [False, True])
@pytest.mark.parametrize("in_dtype", [F16, BF16, F32])
@pytest.mark.parametrize("out_dtype", [F16, BF16, E4M3, E5M2])
@pytest.mark.parametrize("shape", [(32, 128), (96, 320 + 64), (64, 1024)])
def test_magnitude_compress(cuda, shape, in_dtype, out_dtype, col_major):
    import sparse
    w = randn(shape, in_dtype, 11, ties=(shape[0] == 96))
    want_v, want_m = oracle.compress24(w, out_dtype=out_dtype)
    s = sparse.to_sparse_semi_structured(maybe_t(w.to(cuda), col_major), dtype=out_dtype)
    assert s.shape == w.shape and s.dtype == out_dtype
    assert_same(s.values(), want_v, "values")
    assert_same(s.indices(), want_m, "meta")
    assert_same(s.to_dense(), oracle.decompress24(want_v, want_m), "to_dense")


@pytest.mark.parametrize("out_dtype", [F16, E4M3])
@pytest.mark.parametrize("col_major", [False, True])
def test_canonical_and_panel_storage_agree(cuda, out_dtype, col_major):
    """The same tensor compressed into the canonical and into the panel layout: identical
    values()/indices()/to_dense() and identical products."""
    import sparse
    cls = sparse.SparseSemiStructuredTensor
    w = randn((96, 384), F16, 18)
    x = randn((40 if out_dtype == F16 else 48, 384), F16, 19).to(cuda)
    want_v, want_m = oracle.compress24(w, out_dtype=out_dtype)
    outs = []
    try:
        for panel in (True, False):
            cls._PANEL_LAYOUT = panel
            s = sparse.to_sparse_semi_structured(maybe_t(w.to(cuda), col_major), dtype=out_dtype)
            assert s._store_layout == (1 if panel else 0)
            assert_same(s.values(), want_v, f"values panel={panel}")
            assert_same(s.indices(), want_m, f"meta panel={panel}")
            assert_same(s.to_dense(), oracle.decompress24(want_v, want_m), f"to_dense panel={panel}")
            outs.append(torch.mm(x.to(out_dtype), s.t()))
            outs.append(torch.mm(s, x.to(out_dtype).t().contiguous()))
    finally:
        cls._PANEL_LAYOUT = True
    assert_same(outs[0], outs[2], "x.W^T panel vs canonical")
    assert_same(outs[1], outs[3], "W.x^T panel vs canonical")
    # round trip through the canonical constructor arguments
    s2 = cls(None, original_shape=s.shape, sparse_tensor_cutlass=s.values(), meta_tensor_cutlass=s.indices(), dtype=out_dtype)
    assert_same(torch.mm(x.to(out_dtype), s2.t()), outs[0], "rebuilt from canonical pieces")


def test_docstring_known_answer(cuda):
    import sparse
    a = torch.tensor([0.0, 0.0, 1.0, 1.0]).tile((128, 32)).half().to(cuda)
    s = sparse.to_sparse_semi_structured(a)
    assert s.values().eq(1).all() and s.values().shape == (128, 64)
    assert s.indices().eq(-4370).all() and s.indices().dtype == torch.int16
    assert s.indices_cutlass().eq(-4370).all()


def test_config1_compress_and_mm(cuda):
    """BASELINE config 1 (the reference's CPU-runnable case), on the GPU path."""
    import sparse
    g = torch.Generator().manual_seed(0)
    w = (0.02 * torch.randn(3072, 768, generator=g)).half()
    x = torch.randn(12288, 768, generator=g)
    want_v, want_m = oracle.compress24(w)
    s = sparse.to_sparse_semi_structured(w.to(cuda))
    assert_same(s.values(), want_v, "values")
    assert_same(s.indices(), want_m, "meta")
    mask = oracle.prune24_mask(w)
    ref = oracle.spmm_ref(x.half(), torch.where(mask, w, torch.zeros_like(w)))
    out = torch.mm(x.half().to(cuda), s.t()).float().cpu()
    rel = (out - ref).norm() / ref.norm()
    assert out.shape == (12288, 3072) and rel < 1e-2, rel


@pytest.mark.parametrize("col_major", [False, True])
@pytest.mark.parametrize("mask_dtype", [torch.bool, F16, F32])
@pytest.mark.parametrize("in_dtype,out_dtype", [(F32, F16), (F16, F16), (BF16, BF16), (F32, E4M3)])
def test_mask_compress(cuda, in_dtype, out_dtype, mask_dtype, col_major):
    import sparse
    w = randn((64, 256), in_dtype, 12)
    _, mask = oracle.transposable_mask(w.float())
    g = torch.Generator().manual_seed(13)
    mask[:8] = torch.rand(8, 256, generator=g) < 0.5            # invalid groups follow the truth table
    mask = mask.to(mask_dtype)
    want_v, want_m = oracle.compress24(w, mask=mask, out_dtype=out_dtype)
    s = sparse.to_sparse_semi_structured(maybe_t(w.to(cuda), col_major), mask=maybe_t(mask.to(cuda), col_major), dtype=out_dtype)
    assert_same(s.values(), want_v, "values")
    assert_same(s.indices(), want_m, "meta")


@pytest.mark.parametrize("mask_dtype", [torch.bool, BF16, F32])
@pytest.mark.parametrize("in_dtype,out_dtype,shape", [
    (F32, F16, (64, 64)), (F32, F16, (192, 320)), (F16, F16, (128, 448)), (BF16, BF16, (320, 128)),
    (F32, E4M3, (128, 384)), (BF16, E5M2, (256, 128))])
def test_mask_compress_pair(cuda, in_dtype, out_dtype, mask_dtype, shape):
    """W and W^T compressed from one read: each result must carry the bytes of the separate
    conversion of w / w.T (oracle), for transposable masks and for invalid groups."""
    import sparse
    from sparse import _native as N
    w = randn(shape, in_dtype, 15)
    _, mask = oracle.transposable_mask(w.float())
    g = torch.Generator().manual_seed(16)
    mask[:8] = torch.rand(8, shape[1], generator=g) < 0.5        # groups with 0..4 kept elements, both directions
    mask = mask.to(mask_dtype)
    want_v, want_m = oracle.compress24(w, mask=mask, out_dtype=out_dtype)
    want_vt, want_mt = oracle.compress24(w.t().contiguous(), mask=mask.t().contiguous(), out_dtype=out_dtype)
    s, s_t = sparse.to_sparse_semi_structured_pair(w.to(cuda), mask.to(cuda), dtype=out_dtype)
    assert s.shape == shape and s_t.shape == shape[::-1]
    assert s._store_layout == N.COMPRESSED_PANEL and s_t._store_layout == N.COMPRESSED_PANEL
    assert_same(s.values(), want_v, "values")
    assert_same(s.indices(), want_m, "meta")
    assert_same(s_t.values(), want_vt, "values of the transpose")
    assert_same(s_t.indices(), want_mt, "meta of the transpose")
    # canonical output through the C entry point, with padded rows of the dense matrix and the mask
    m, k = shape
    wide = torch.zeros((m, k + 24), dtype=in_dtype, device=cuda)
    wide[:, 8:8 + k] = w.to(cuda)
    mk = mask.to(cuda)
    mk = mk.view(torch.uint8) if mk.dtype == torch.bool else mk
    mwide = torch.zeros((m, k + 16), dtype=mk.dtype, device=cuda)
    mwide[:, 16:] = mk
    wv, mv = wide[:, 8:8 + k], mwide[:, 16:]
    idt = torch.int32 if out_dtype in FLOAT8 else torch.int16
    cv = torch.empty((m, k // 2), dtype=out_dtype, device=cuda)
    cvt = torch.empty((k, m // 2), dtype=out_dtype, device=cuda)
    cm = torch.empty((m, k // 8), dtype=torch.uint8, device=cuda)
    cmt = torch.empty((k, m // 8), dtype=torch.uint8, device=cuda)
    N.check(N.lib().tf24_prune_compress_dual(
        wv.data_ptr(), N.dtype_code(in_dtype), wv.stride(0), m, k, mv.data_ptr(), N.dtype_code(mv.dtype), mv.stride(0),
        cv.data_ptr(), cm.data_ptr(), cvt.data_ptr(), cmt.data_ptr(), N.dtype_code(out_dtype), N.COMPRESSED_CANONICAL, N.stream_ptr()))
    assert_same(cv, want_v)
    assert_same(cm.view(idt), want_m)
    assert_same(cvt, want_vt)
    assert_same(cmt.view(idt), want_mt)


def test_mask_compress_pair_falls_back_and_rejects(cuda):
    """Shapes only one direction supports run the two separate conversions (and raise where those
    raise); the C entry point refuses them."""
    import sparse
    from sparse import _native as N
    w = randn((96, 128), F16, 17)                               # 96 rows: fine for w, not for w.T (needs % 64)
    mask = oracle.prune24_mask(w)
    with pytest.raises(RuntimeError):
        sparse.to_sparse_semi_structured_pair(w.to(cuda), mask.to(cuda))
    wt = randn((128, 192), F16, 18).t()                         # column-major input: separate conversions, same bytes
    _, mask = oracle.transposable_mask(wt.contiguous().float())
    s, s_t = sparse.to_sparse_semi_structured_pair(wt.to(cuda), mask.to(cuda))
    want_v, want_m = oracle.compress24(wt.contiguous(), mask=mask)
    want_vt, want_mt = oracle.compress24(wt.t().contiguous(), mask=mask.t().contiguous())
    assert_same(s.values(), want_v)
    assert_same(s.indices(), want_m)
    assert_same(s_t.values(), want_vt)
    assert_same(s_t.indices(), want_mt)
    lib = N.lib()
    assert lib.tf24_prune_compress_dual_validate(N.F16, 128, 96, 128, N.U8, 128, N.F16, N.COMPRESSED_PANEL) != 0
    assert lib.tf24_prune_compress_dual_validate(N.F16, 128, 128, 128, N.U8, 128, N.E4M3, N.COMPRESSED_PANEL) == 0
    assert lib.tf24_prune_compress_dual_validate(N.F16, 64, 128, 64, N.U8, 64, N.E4M3, N.COMPRESSED_PANEL) != 0
    assert lib.tf24_prune_compress_dual_validate(N.F16, 120, 128, 128, N.U8, 128, N.F16, N.COMPRESSED_PANEL) != 0   # ld < k
    assert lib.tf24_prune_compress_dual_validate(N.U8, 128, 128, 128, N.U8, 128, N.F16, N.COMPRESSED_PANEL) != 0


@pytest.mark.parametrize("mode", ["magnitude", "mvue"])
@pytest.mark.parametrize("dtype,shape", [(F16, (96, 320)), (BF16, (64, 128)), (F32, (160, 192)), (F16, (3072, 1024))])
def test_compress_with_row_sums(cuda, dtype, shape, mode):
    """Compression of a column-major matrix that also returns its row sums (the bias gradient when the
    matrix is dY^T): compressed bytes identical to the plain conversion, sums within float32
    accumulation error of the exact sum and one rounding to the input dtype."""
    import sparse
    from sparse import _native as N
    m, k = shape
    t = randn((k, m), dtype, 19).t()                             # [m, k] column-major
    rand = torch.rand((k // 2, m), generator=torch.Generator().manual_seed(20)).t() if mode == "mvue" else None
    kw = dict(MVUE24=mode == "mvue", dtype=F16, rand=None if rand is None else rand.to(cuda))
    plain = sparse.to_sparse_semi_structured(t.to(cuda), **kw)
    fused, sums = sparse.to_sparse_semi_structured_with_row_sums(t.to(cuda), **kw)
    assert fused._store_layout == N.COMPRESSED_PANEL
    assert_same(fused.values(), plain.values().cpu(), "values")
    assert_same(fused.indices(), plain.indices().cpu(), "meta")
    want = t.double().sum(1)
    assert sums.shape == (m,) and sums.dtype == dtype
    eps = {F16: 2.0 ** -11, BF16: 2.0 ** -8, F32: 2.0 ** -24}[dtype]
    tol = eps * want.abs() + 2e-7 * (k ** 0.5) * t.double().abs().sum(1) / k ** 0.5 + 1e-30
    assert ((sums.double().cpu() - want).abs() <= tol + eps * want.abs().max()).all()
    # deterministic: the same bits every time
    again = sparse.to_sparse_semi_structured_with_row_sums(t.to(cuda), **kw)[1]
    assert again.equal(sums)


def test_compress_with_row_sums_other_layouts(cuda):
    """Row-major input runs the two operations separately; the C entry point refuses it."""
    import sparse
    from sparse import _native as N
    t = randn((64, 128), F16, 21)
    s, sums = sparse.to_sparse_semi_structured_with_row_sums(t.to(cuda))
    want_v, want_m = oracle.compress24(t)
    assert_same(s.values(), want_v)
    assert_same(s.indices(), want_m)
    assert torch.allclose(sums.float().cpu(), t.float().sum(1), rtol=2e-3, atol=2e-2)
    d = t.to(cuda)
    v = torch.empty(64 * 64, dtype=F16, device=cuda)
    mt = torch.empty(64 * 16, dtype=torch.uint8, device=cuda)
    out = torch.empty(64, dtype=F16, device=cuda)
    ws = torch.empty(64, dtype=torch.float32, device=cuda)
    call = lambda layout, ws_bytes: N.lib().tf24_prune_compress_rowsum(
        d.data_ptr(), N.F16, layout, 128, 64, 128, N.PRUNE_MAGNITUDE, None, N.U8, 0, None, 0, v.data_ptr(), N.F16, mt.data_ptr(),
        N.COMPRESSED_PANEL, out.data_ptr(), N.F16, ws.data_ptr(), ws_bytes, N.stream_ptr())
    assert call(N.ROW_MAJOR, 256) == -5
    assert N.lib().tf24_prune_compress_rowsum_workspace_bytes(64, 128) == 256
    assert N.lib().tf24_prune_compress_rowsum_workspace_bytes(3072, 12288) == 96 * 3072 * 4


def test_mask_layout_mismatch_is_copied(cuda):
    import sparse
    w = randn((64, 128), F16, 14)
    mask = oracle.prune24_mask(w)
    want_v, want_m = oracle.compress24(w, mask=mask)
    # column-major dense with a row-major mask and vice versa
    s1 = sparse.to_sparse_semi_structured(maybe_t(w.to(cuda), True), mask=mask.to(cuda))
    s2 = sparse.to_sparse_semi_structured(w.to(cuda), mask=maybe_t(mask.to(cuda), True))
    for s in (s1, s2):
        assert_same(s.values(), want_v)
        assert_same(s.indices(), want_m)


@pytest.mark.parametrize("col_major", [False, True])
@pytest.mark.parametrize("in_dtype,out_dtype", [(BF16, F16), (F16, F16), (F32, BF16), (BF16, E4M3), (F32, E4M3), (F32, E5M2)])
@pytest.mark.parametrize("shape", [(32, 128), (128, 640)])
def test_mvue_compress(cuda, shape, in_dtype, out_dtype, col_major):
    import sparse
    w = randn(shape, in_dtype, 15)
    w[0, :8] = 0                                                 # degenerate all-zero groups
    u = torch.rand(shape, generator=torch.Generator().manual_seed(16))
    u[1, 1] = 0.0                                                # r1 == 0: a single element may be kept
    want_v, want_m, _ = oracle.mvue24(w, u, out_dtype=out_dtype)
    s = sparse.to_sparse_semi_structured(maybe_t(w.to(cuda), col_major), MVUE24=True, rand=maybe_t(u.to(cuda), col_major), dtype=out_dtype)
    assert_same(s.values(), want_v, "values")
    assert_same(s.indices(), want_m, "meta")


@pytest.mark.parametrize("col_major", [False, True])
@pytest.mark.parametrize("out_dtype", [F16, E4M3])
def test_mvue_compress_packed_uniforms(cuda, out_dtype, col_major):
    """A [m, k/2] uniform tensor holds exactly the uniforms the estimator uses: group g of a row
    takes columns 2g and 2g+1.  Same result as the full-shape tensor carrying them in columns 4g, 4g+1."""
    import sparse
    shape = (64, 384)
    w = randn(shape, BF16, 25)
    up = torch.rand((shape[0], shape[1] // 2), generator=torch.Generator().manual_seed(26))
    full = torch.full(shape, 0.5)
    full[:, 0::4], full[:, 1::4] = up[:, 0::2], up[:, 1::2]
    want_v, want_m, _ = oracle.mvue24(w, full, out_dtype=out_dtype)
    s = sparse.to_sparse_semi_structured(maybe_t(w.to(cuda), col_major), MVUE24=True, rand=maybe_t(up.to(cuda), col_major), dtype=out_dtype)
    assert_same(s.values(), want_v, "values")
    assert_same(s.indices(), want_m, "meta")
    with pytest.raises(RuntimeError):
        sparse.to_sparse_semi_structured(w.to(cuda), MVUE24=True, rand=up[:, :-8].to(cuda), dtype=out_dtype)


@pytest.mark.parametrize("col_major", [False, True])
@pytest.mark.parametrize("in_dtype,out_dtype,shape", [(BF16, F16, (64, 128)), (F16, F16, (96, 320)), (F32, BF16, (32, 64)), (F16, E4M3, (64, 256))])
def test_mvue_seeded_uniforms(cuda, in_dtype, out_dtype, shape, col_major):
    """Uniforms generated inside the kernel: tf24_mvue_uniforms writes the oracle's Philox stream, and
    compressing with rand=(seed, offset) gives the bytes of compressing with that tensor supplied."""
    import sparse
    from sparse import _native as N
    m, k = shape
    seed, offset = 0x1234567890abcdef, 40
    want_u = oracle.mvue_uniforms(seed, offset, m, k)
    got = torch.empty((m, k // 2), dtype=torch.float32, device=cuda)
    N.check(N.lib().tf24_mvue_uniforms(seed, offset, m, k, N.ROW_MAJOR, got.data_ptr(), k // 2, N.stream_ptr()))
    assert got.cpu().equal(want_u)
    got_t = torch.empty((k // 2, m), dtype=torch.float32, device=cuda)
    N.check(N.lib().tf24_mvue_uniforms(seed, offset, m, k, N.COL_MAJOR, got_t.data_ptr(), m, N.stream_ptr()))
    assert got_t.t().cpu().equal(want_u)
    w = randn(shape, in_dtype, 23)
    full = torch.zeros(shape)
    full[:, 0::4], full[:, 1::4] = want_u[:, 0::2], want_u[:, 1::2]
    want_v, want_m, _ = oracle.mvue24(w, full, out_dtype=out_dtype)
    wd = maybe_t(w.to(cuda), col_major)
    s = sparse.to_sparse_semi_structured(wd, MVUE24=True, dtype=out_dtype, rand=(seed, offset))
    assert_same(s.values(), want_v, "values")
    assert_same(s.indices(), want_m, "meta")
    if col_major and out_dtype not in FLOAT8:
        s2, sums = sparse.to_sparse_semi_structured_with_row_sums(wd, MVUE24=True, dtype=out_dtype, rand=(seed, offset))
        assert_same(s2.values(), want_v)
        assert_same(s2.indices(), want_m)


def test_mvue_default_sampling_follows_torch_seed(cuda):
    """Without `rand` the (seed, offset) pair comes from torch's generator: torch.manual_seed makes the
    sampling reproducible, successive calls draw different uniforms, two values are kept per group."""
    import sparse
    w = randn((64, 256), F16, 24).to(cuda)
    torch.manual_seed(77)
    a1 = sparse.to_sparse_semi_structured(w, MVUE24=True)
    a2 = sparse.to_sparse_semi_structured(w, MVUE24=True)
    torch.manual_seed(77)
    b1 = sparse.to_sparse_semi_structured(w.t().contiguous().t(), MVUE24=True)      # same matrix, column-major storage
    assert a1.indices().equal(b1.indices()) and a1.values().equal(b1.values())
    assert not a1.indices().equal(a2.indices())
    dense = a1.to_dense()
    assert ((dense != 0).view(64, 64, 4).sum(-1) <= 2).all()
    # unbiased: the mean over many draws approaches w
    acc = torch.zeros_like(w, dtype=torch.float32)
    for _ in range(200):
        acc += sparse.to_sparse_semi_structured(w, MVUE24=True).to_dense().float()
    err = (acc / 200 - w.float()).abs().mean() / w.float().abs().mean()
    assert err < 0.12, err


@pytest.mark.parametrize("out_dtype", [F16, BF16, E4M3, E5M2])
@pytest.mark.parametrize("in_dtype,shape,extra", [(BF16, (64, 128), 0), (F16, (96, 384), 8), (F32, (32, 2176), 64), (F32, (1056, 256), 0), (BF16, (160, 640), 24)])
def test_mvue_panel_conversion(cuda, in_dtype, out_dtype, shape, extra):
    """The kernel for row-major input and panel output: 16 rows x 128 columns to a block, rows of the matrix longer than its columns,
    uniforms from every source, groups whose largest element outweighs the others by up to 2^26 -- the bits of the oracle."""
    import sparse
    m, k = shape
    g = torch.Generator().manual_seed(m + k)
    wide = (torch.randn((m, k + extra), generator=g) * torch.exp2(torch.randint(-12, 15 if in_dtype != F16 else 4, (m, k + extra), generator=g).float())).to(in_dtype)
    w = wide[:, :k]
    seed, offset = 0xfedcba9876543210, (1 << 33) + 12
    packed = oracle.mvue_uniforms(seed, offset, m, k)
    full = torch.zeros(shape)
    full[:, 0::4], full[:, 1::4] = packed[:, 0::2], packed[:, 1::2]
    want_v, want_m, _ = oracle.mvue24(w, full, out_dtype=out_dtype)
    for rand in ((seed, offset), packed.to(cuda), full.to(cuda)):
        s = sparse.to_sparse_semi_structured(wide.to(cuda)[:, :k], MVUE24=True, dtype=out_dtype, rand=rand)
        assert_same(s.indices(), want_m, "meta")
        assert_same(torch.nan_to_num(s.values().float().cpu(), 1.5), torch.nan_to_num(want_v.float(), 1.5), "values")


@pytest.mark.parametrize("out_dtype", [F16, BF16])
@pytest.mark.parametrize("in_dtype,shape,extra", [(F16, (64, 192), 0), (F32, (32, 64), 0), (BF16, (96, 1088), 8)])
def test_mvue_panel_conversion_with_partial_blocks(cuda, in_dtype, out_dtype, shape, extra):
    """Half a block on the right: an odd multiple of 64 columns, which only 16-bit values take."""
    test_mvue_panel_conversion(cuda, in_dtype, out_dtype, shape, extra)


def _wide_range(shape, seed):
    """float32 values whose exponents span denormals to 2^60, with zeros, negative zeros and groups
    dominated by one element (sum - a_i rounds to zero): operands the in-range division must hand
    to the general one."""
    g = torch.Generator().manual_seed(seed)
    expo = torch.randint(-140, 61, shape, generator=g).float()
    w = torch.randn(shape, generator=g) * torch.exp2(expo)
    flat = w.view(-1, 4)
    flat[0::7, 1] = 0.0
    flat[3::7, 2] = -0.0
    flat[5::11] = torch.tensor([1.0e6, 1.0e-7, 0.0, -1.0e-7])
    flat[6::13] = torch.tensor([3.0e38, 1.0, -2.0e38, 1.0e-30])
    return w


@pytest.mark.parametrize("col_major", [False, True])
def test_mvue_wide_dynamic_range(cuda, col_major):
    import sparse
    w = _wide_range((64, 256), 18)
    u = torch.rand(w.shape, generator=torch.Generator().manual_seed(19))
    want = oracle.mvue24_dense(w, u)
    got = sparse.MVUE24_approx_triton(maybe_t(w.to(cuda), col_major), rand=maybe_t(u.to(cuda), col_major)).cpu()
    assert torch.equal(got.isnan(), want.isnan())
    ok = ~want.isnan()
    assert_same(torch.where(ok, got, torch.zeros(())), torch.where(ok, want, torch.zeros(())), "mvue dense, wide range")
    want_v, want_m, _ = oracle.mvue24(w, u, out_dtype=BF16)
    s = sparse.to_sparse_semi_structured(maybe_t(w.to(cuda), col_major), MVUE24=True, rand=maybe_t(u.to(cuda), col_major), dtype=BF16)
    assert_same(s.indices(), want_m, "meta")
    gv = s.values().cpu()
    assert torch.equal(gv.isnan(), want_v.isnan())
    okv = ~want_v.isnan()
    assert_same(torch.where(okv, gv, torch.zeros((), dtype=BF16)), torch.where(okv, want_v, torch.zeros((), dtype=BF16)), "values, wide range")


def test_mvue_default_rand_keeps_two(cuda):
    import sparse
    w = randn((64, 128), F16, 17).to(cuda)
    torch.manual_seed(0)
    s = sparse.to_sparse_semi_structured(w, MVUE24=True)
    dense = s.to_dense()
    assert (dense != 0).reshape(-1, 4).sum(-1).le(2).all()


def test_compress_errors(cuda):
    import sparse
    with pytest.raises(RuntimeError):
        sparse.to_sparse_semi_structured(torch.zeros(32, 64, dtype=F16))                       # not on the GPU
    with pytest.raises(RuntimeError):
        sparse.to_sparse_semi_structured(torch.zeros(2, 32, 64, dtype=F16, device=cuda))       # not 2-d
    with pytest.raises(RuntimeError):
        sparse.to_sparse_semi_structured(torch.zeros(32, 64, dtype=F16, device=cuda), dtype=torch.float64)
    with pytest.raises(RuntimeError):
        sparse.to_sparse_semi_structured(torch.zeros(48, 64, dtype=F16, device=cuda))
    with pytest.raises(RuntimeError):
        sparse.to_sparse_semi_structured(torch.zeros(32, 64, dtype=F16, device=cuda), dtype=E4M3)  # needs k % 128
    with pytest.raises(RuntimeError):
        sparse.to_sparse_semi_structured(torch.zeros(32, 64, dtype=F16, device=cuda), MVUE24=True,
                                         mask=torch.ones(32, 64, dtype=torch.bool, device=cuda))


# ------------------------------------------------------------------ transposable search
@pytest.mark.parametrize("col_major", [False, True])
@pytest.mark.parametrize("use_abs", [True, False])
@pytest.mark.parametrize("dtype", [F16, BF16, F32])
@pytest.mark.parametrize("ties", [False, True])
def test_transposable(cuda, dtype, use_abs, col_major, ties):
    import sparse
    w = randn((96, 192), dtype, 21, ties=ties)
    if ties:
        w[:4, :8] = 0
        w[4:8, :4] = 1
    want_s, want_m = oracle.transposable_mask(w, use_abs=use_abs)
    got_s, got_m = sparse.TransposableSparse(abs=use_abs)(maybe_t(w.to(cuda), col_major))
    assert got_m.dtype == torch.bool
    assert_same(got_m, want_m, "mask")
    assert_same(got_s, want_s, "sparse")
    if ties or dtype != F32:
        _, brute, _ = oracle.transposable_mask_bruteforce(w, use_abs=use_abs)
        if ties:
            assert_same(got_m, brute, "mask vs 90-way brute force")


def test_transposable_errors(cuda):
    import sparse
    ts = sparse.TransposableSparse()
    for shape in [(33, 64), (32, 32)]:
        with pytest.raises(RuntimeError):
            ts(torch.zeros(shape, device=cuda))
    with pytest.raises(RuntimeError):
        ts(torch.zeros(32, 64, dtype=torch.float64, device=cuda))
    with pytest.raises(RuntimeError):
        ts(torch.zeros(2, 32, 64, device=cuda))


# ------------------------------------------------------------------ dense-shaped operators
@pytest.mark.parametrize("col_major", [False, True])
@pytest.mark.parametrize("dtype", [F16, BF16, F32])
def test_soft_threshold(cuda, dtype, col_major):
    import sparse
    w = randn((64, 256), dtype, 31, ties=(dtype == F16))
    want_s, want_m = oracle.soft_threshold24(w)
    got_s, got_m = sparse.soft_threshold24_triton(maybe_t(w.to(cuda), col_major))
    assert_same(got_s, want_s, "sparse")
    assert_same(got_m, want_m, "mask")
    assert got_s.stride() == maybe_t(w, col_major).stride()


@pytest.mark.parametrize("col_major", [False, True])
@pytest.mark.parametrize("dtype", [F16, BF16, F32])
def test_sparse24_and_mvue_dense(cuda, dtype, col_major):
    import sparse
    w = randn((64, 256), dtype, 32)
    want_s, want_m = oracle.sparse24_dense(w)
    got_s, got_m = sparse.sparse24_triton(maybe_t(w.to(cuda), col_major))
    assert_same(got_s, want_s, "sparse24")
    assert_same(got_m, want_m, "mask24")
    u = torch.rand(w.shape, generator=torch.Generator().manual_seed(33))
    got = sparse.MVUE24_approx_triton(maybe_t(w.to(cuda), col_major), rand=maybe_t(u.to(cuda), col_major))
    assert_same(got, oracle.mvue24_dense(w, u), "mvue dense")


# ------------------------------------------------------------------ masked decay
@pytest.mark.parametrize("gdt,pdt,mdt", [(F32, F32, torch.bool), (F32, BF16, torch.bool), (F32, F32, F32),
                                         (BF16, BF16, BF16), (F16, F32, torch.uint8)])
@pytest.mark.parametrize("n", [(64, 64), (7, 13), (1000003,)])
def test_masked_add(cuda, gdt, pdt, mdt, n):
    import sparse
    g = torch.Generator().manual_seed(41)
    grad = (1e-3 * torch.randn(n, generator=g)).to(gdt)
    p = torch.randn(n, generator=g).to(pdt)
    mask = (torch.rand(n, generator=g) < 0.5).to(mdt)
    want = oracle.masked_add(grad, p, mask, alpha=2e-4)
    gg = grad.to(cuda)
    assert sparse.masked_add_(gg, p.to(cuda), mask.to(cuda), alpha=2e-4) is None
    assert_same(gg, want)


def test_masked_add_reference_vector(cuda):
    import sparse
    grad = torch.tensor([1.0, 1.0, 1.0, 1.0], device=cuda)
    sparse.masked_add_(grad, torch.tensor([1.0, 2.0, 3.0, 4.0], device=cuda), torch.tensor([1.0, 0.0, 1.0, 0.0], device=cuda), alpha=0.03)
    assert torch.allclose(grad.cpu(), torch.tensor([1.0, 1.06, 1.0, 1.12]), atol=1e-7)


# ------------------------------------------------------------------ 2:4 matmul
def _small_ints(shape, seed, lo=-3, hi=4):
    return torch.randint(lo, hi, shape, generator=torch.Generator().manual_seed(seed)).float()


@pytest.mark.parametrize("dtype", [F16, BF16, E4M3, E5M2])
@pytest.mark.parametrize("dims", [(32, 128, 16), (64, 256, 40), (96, 384, 200), (160, 1024, 72)])
def test_spmm_exact_small_integers(cuda, dtype, dims):
    """Small-integer operands: every product and partial sum is exact in float32, so the
    result must EQUAL the dense masked product -- pins operand and index layout."""
    import sparse
    n, k, m = dims
    if dtype in FLOAT8 and m % 16:
        m += 8
    w = _small_ints((n, k), 51).to(dtype)
    x = _small_ints((m, k), 52).to(dtype)
    mask = oracle.prune24_mask(w.float())
    ref = oracle.spmm_ref(x.float(), torch.where(mask, w.float(), torch.zeros(())))
    s = sparse.to_sparse_semi_structured(w.float().to(cuda), dtype=dtype)
    out = torch.mm(x.to(cuda), s.t())                      # second operand sparse: x . W^T
    assert out.shape == (m, n)
    assert out.dtype == (torch.float32 if dtype in FLOAT8 else dtype)
    ref = ref.to(out.dtype).float()                        # the kernel rounds the exact sum once
    assert out.float().cpu().equal(ref)
    # first operand sparse: W . B with B [k, j] row-major (k strided) and as a transposed view
    b = x.t().contiguous()
    out2 = torch.mm(s, b.to(cuda))
    assert out2.shape == (n, m) and out2.float().cpu().equal(ref.t())
    out3 = torch.mm(s, x.to(cuda).t())
    assert out3.float().cpu().equal(ref.t())
    # second operand sparse with a column-major x
    out4 = torch.mm(maybe_t(x.to(cuda), True), s.t())
    assert out4.float().cpu().equal(ref)


@pytest.mark.parametrize("dtype,tol", [(F16, 1e-2), (BF16, 1e-2), (E4M3, 5e-2), (E5M2, 5e-2)])
def test_spmm_random_tolerance(cuda, dtype, tol):
    import sparse
    n, k, m = 256, 512, 328 if dtype not in FLOAT8 else 336
    w = randn((n, k), F32, 53, scale=0.02)
    x = randn((m, k), F32, 54)
    if dtype in FLOAT8:
        sw, sx = 448.0 / w.abs().max(), 448.0 / x.abs().max()
        wq, xq = (w * sw).to(dtype), (x * sx).to(dtype)
    else:
        sw = sx = 1.0
        wq, xq = w.to(dtype), x.to(dtype)
    mask = oracle.prune24_mask(wq.float())
    ref = oracle.spmm_ref(xq.float(), torch.where(mask, wq.float(), torch.zeros(())))
    s = sparse.to_sparse_semi_structured(wq.float().to(cuda), dtype=dtype)
    out = torch.mm(xq.to(cuda), s.t()).float().cpu()
    rel = (out - ref).norm() / ref.norm()
    assert rel < tol, rel


def test_spmm_bias_linear_padding(cuda):
    import sparse
    n, k, m = 64, 128, 21                                   # m is padded to 24 and sliced back
    w = _small_ints((n, k), 55).half()
    x = _small_ints((3, 7, k), 56).half()
    bias = _small_ints((n,), 57).half()
    mask = oracle.prune24_mask(w)
    wm = torch.where(mask, w, torch.zeros_like(w))
    s = sparse.to_sparse_semi_structured(w.to(cuda))
    ref = oracle.linear_ref(x, wm, bias)
    out = torch.nn.functional.linear(x.to(cuda), s, bias.to(cuda))
    assert out.shape == (3, 7, n) and out.float().cpu().equal(ref)
    out = torch.addmm(bias.to(cuda), x.reshape(m, k).to(cuda), s.t())
    assert out.float().cpu().equal(ref.reshape(m, n))
    with torch.inference_mode():
        out = torch.nn.functional.linear(x.to(cuda), s, bias.to(cuda))
    assert out.float().cpu().equal(ref)


def test_dispatch_rules(cuda):
    import sparse
    w = _small_ints((32, 64), 58).half().to(cuda)
    s = sparse.to_sparse_semi_structured(w)
    assert s.t().transposed and s.t().shape == (64, 32) and not s.t().t().transposed
    assert s.detach()._store_values.data_ptr() == s._store_values.data_ptr()
    x = torch.ones(8, 64, dtype=F16, device=cuda)
    with pytest.raises(NotImplementedError):
        torch.mm(x, s)                                     # second operand must be transposed
    with pytest.raises(NotImplementedError):
        torch.mm(s.t(), x.t())                             # first operand must not be
    with pytest.raises(NotImplementedError):
        s + 1


@pytest.mark.parametrize("dtype,k", [(F16, 256), (F16, 320), (BF16, 704), (E4M3, 512), (E4M3, 640)])
def test_spmm_chained_tiles_with_partial_edges(cuda, dtype, k):
    """More 256 x 256 tiles than compute units: one workgroup per compute unit chains its tiles (the next
    tile's first copies ride in the current tile's last two stages).  17 x 17 tiles with partial last
    row and column of tiles, from the shortest k the chained form takes (4 stages) up; exact on small
    integers, with and without bias, against the float32 product; 16-bit and 8-bit operands."""
    import sparse
    n, m = 4128, 4112
    odt = torch.bfloat16 if dtype in FLOAT8 else dtype
    w = _small_ints((n, k), 71, -2, 3).to(dtype)
    x = _small_ints((m, k), 72, -2, 3).to(dtype)
    bias = _small_ints((n,), 73).to(odt)
    mask = oracle.prune24_mask(w.float())
    ref = oracle.spmm_ref(x.float(), torch.where(mask, w.float(), torch.zeros(())))
    s = sparse.to_sparse_semi_structured(w.float().to(cuda), dtype=dtype)
    xg = x.to(cuda)
    out = sparse.sparse_semi_structured_linear(xg, s, out_dtype=odt)
    assert out.shape == (m, n) and out.float().cpu().equal(ref.to(odt).float())
    out = sparse.sparse_semi_structured_linear(xg, s, bias_opt=bias.to(cuda), out_dtype=odt)
    assert out.float().cpu().equal((ref + bias.float()).to(odt).float())
    # twice in a row on the same buffers: nothing left over from the first launch
    again = sparse.sparse_semi_structured_linear(xg, s, bias_opt=bias.to(cuda), out_dtype=odt)
    assert again.equal(out)


@pytest.mark.parametrize("dtype,k,act,scale", [(F16, 256, "relu", 0.5), (BF16, 320, "relu", 1.0), (E4M3, 512, "relu", 0.25),
                                               (F16, 320, "silu", 0.5), (BF16, 256, "gelu", 1.0), (E4M3, 640, "gelu", 0.125),
                                               (F16, 256, "gelu", 1.0), (E5M2, 512, "silu", 1.0)])
def test_spmm_chained_tiles_activation_and_scale(cuda, dtype, k, act, scale):
    """The chained-tile kernel's output passes with an activation (the bias of a wave's rows reaches them through
    LDS; zeros without a bias): 17 x 17
    tiles of 256 x 256 with partial edge tiles, more tiles than compute units.  Scale and bias act on exact
    float32 sums of small integers, so ReLU results are exact (one rounding of an exact value); SiLU and
    GELU are compared with torch's float32 functions of the same exact argument within 2e-3 + one unit in
    the last place of the 16-bit output (the kernel's exp / erf differ from torch's by a few float32 ulps)."""
    import sparse
    n, m = 4128, 4112
    odt = torch.bfloat16 if dtype in FLOAT8 else dtype
    w = _small_ints((n, k), 74, -2, 3).to(dtype)
    x = _small_ints((m, k), 75, -2, 3).to(dtype)
    bias = (_small_ints((n,), 76) * 0.5).to(odt)
    mask = oracle.prune24_mask(w.float())
    pre = oracle.spmm_ref(x.float(), torch.where(mask, w.float(), torch.zeros(()))) * scale + bias.float()
    s = sparse.to_sparse_semi_structured(w.float().to(cuda), dtype=dtype)
    out = sparse.sparse_semi_structured_linear(x.to(cuda), s, bias_opt=bias.to(cuda), activation_opt=act, out_dtype=odt, scale=scale)
    assert out.shape == (m, n) and out.dtype == odt
    got = out.float().cpu()
    if act == "relu":
        assert got.equal(pre.clamp_min(0).to(odt).float())
    else:
        want = torch.nn.functional.silu(pre) if act == "silu" else torch.nn.functional.gelu(pre)
        ulp = 2.0 ** -8 if odt == torch.bfloat16 else 2.0 ** -11
        err = (got - want).abs()
        assert bool((err <= 2e-3 + (2e-3 + ulp) * want.abs()).all()), float(err.max())
    again = sparse.sparse_semi_structured_linear(x.to(cuda), s, bias_opt=bias.to(cuda), activation_opt=act, out_dtype=odt, scale=scale)
    assert again.equal(out)
    # the same activation without a bias, right behind a launch that had one
    nobias = sparse.sparse_semi_structured_linear(x.to(cuda), s, activation_opt=act, out_dtype=odt, scale=scale).float().cpu()
    pre0 = pre - bias.float()
    if act == "relu":
        assert nobias.equal(pre0.clamp_min(0).to(odt).float())
    else:
        want0 = torch.nn.functional.silu(pre0) if act == "silu" else torch.nn.functional.gelu(pre0)
        err0 = (nobias - want0).abs()
        assert bool((err0 <= 2e-3 + (2e-3 + ulp) * want0.abs()).all()), float(err0.max())


@pytest.mark.parametrize("dtype,k,act,n,m", [(F16, 1024, None, 4128, 4112), (BF16, 704, "relu", 4128, 4112),
                                              (E4M3, 1152, "gelu", 4128, 4112), (F16, 576, "silu", 4128, 4112),
                                              (F16, 768, None, 3072, 12288), (E5M2, 2048, None, 4384, 4352),
                                              (F16, 3072, "gelu", 4128, 4112), (BF16, 3136, None, 4128, 4112),
                                              (E4M3, 6144, "relu", 4128, 4112), (E5M2, 6272, "silu", 4384, 4352),
                                              (F16, 2112, "relu", 1760, 12272), (E4M3, 4224, None, 1792, 12288),
                                              (BF16, 2048, "gelu", 2784, 8176), (F16, 2112, None, 800, 12272),
                                              (BF16, 3072, None, 768, 12288), (F16, 2112, None, 4128, 8176),
                                              (E4M3, 4224, "relu", 4128, 8176), (BF16, 2048, None, 4384, 8192)])
def test_spmm_partial_last_round_long_k(cuda, dtype, k, act, n, m):
    """More tiles than compute units with a partial last round and 8 to 49 stages of k (the chained-tile kernel
    with one to three full rounds before the leftover tiles; from 32 stages on in its 4-wave form -- the last three
    shapes but two on 256 x 192 tiles, which need no more rounds there than 256 x 256 ones: 7 x 64 and 11 x 43 tiles with partial edges;
    the next two on 4 x 64 and 3 x 64 such tiles in a single round, where 256 x 256 ones would leave compute units idle;
    the last three with two full rounds of 256 x 256 tiles and one or two more tile rows, which a second launch computes on
    256 x 128 tiles -- in the first two of them the partial row of tiles).  Sums of small integers are exact in float32, so the
    results must equal the oracle's bit for bit, with bias, scale and activation behind the sum, for k contiguous
    and k strided dense operands, on a second call, and through the C ABI without a workspace."""
    import sparse
    odt = torch.bfloat16 if dtype in FLOAT8 else dtype
    w = _small_ints((n, k), 84, -2, 3).to(dtype)
    x = _small_ints((m, k), 85, -2, 3).to(dtype)
    bias = (_small_ints((n,), 86) * 0.5).to(odt)
    mask = oracle.prune24_mask(w.float())
    pre = oracle.spmm_ref(x.float(), torch.where(mask, w.float(), torch.zeros(()))) * 0.5 + bias.float()
    s = sparse.to_sparse_semi_structured(w.float().to(cuda), dtype=dtype)
    xg = x.to(cuda)
    run = lambda xin: sparse.sparse_semi_structured_linear(xin, s, bias_opt=bias.to(cuda), activation_opt=act, out_dtype=odt, scale=0.5)
    out = run(xg)
    got = out.float().cpu()
    if act in (None, "relu"):
        want = pre if act is None else pre.clamp_min(0)
        assert got.equal(want.to(odt).float())
    else:
        want = torch.nn.functional.silu(pre) if act == "silu" else torch.nn.functional.gelu(pre)
        ulp = 2.0 ** -8 if odt == torch.bfloat16 else 2.0 ** -11
        err = (got - want).abs()
        assert bool((err <= 2e-3 + (2e-3 + ulp) * want.abs()).all()), float(err.max())
    assert run(xg).equal(out)
    if dtype not in FLOAT8:
        assert run(maybe_t(xg, True)).equal(out)                # k strided dense operand
    y = torch.empty((m, n), dtype=odt, device=cuda)
    N = sparse._native
    N.check(N.lib().tf24_spmm(s._store_values.data_ptr(), s._store_meta.data_ptr(), s._store_layout, N.operand_code(s._store_values.dtype), n, k,
                              xg.data_ptr(), N.ROW_MAJOR, k, m, y.data_ptr(), N.operand_code(odt), N.COL_MAJOR, n,
                              bias.to(cuda).data_ptr(), 0.5, {None: N.ACT_NONE, "relu": N.ACT_RELU, "silu": N.ACT_SILU, "gelu": N.ACT_GELU}[act],
                              None, 0, N.stream_ptr()))
    assert y.equal(out)


@pytest.mark.parametrize("dtype", [F16, BF16, E4M3, E5M2])
def test_spmm_tiled_all_operand_positions(cuda, dtype):
    """Shapes large enough for the tiled kernel, with partial tiles: both operand positions, both
    layouts of the dense operand, bias, and the i-major / j-major LDS-staged epilogues."""
    import sparse
    n, k, m = 352, 640, 296 if dtype not in FLOAT8 else 304
    odt = torch.float32 if dtype in FLOAT8 else dtype           # 8-bit operands return float32
    w = _small_ints((n, k), 61).to(dtype)
    x = _small_ints((m, k), 62).to(dtype)
    bias = _small_ints((n,), 63).to(odt)
    mask = oracle.prune24_mask(w.float())
    ref = oracle.spmm_ref(x.float(), torch.where(mask, w.float(), torch.zeros(())))
    ref_b = (ref + bias.float()).to(odt).float()
    ref = ref.to(odt).float()
    s = sparse.to_sparse_semi_structured(w.float().to(cuda), dtype=dtype)
    xg = x.to(cuda)
    assert torch.mm(xg, s.t()).float().cpu().equal(ref)                          # k contiguous, j-major store
    assert torch.mm(maybe_t(xg, True), s.t()).float().cpu().equal(ref)           # k strided dense operand
    assert torch.mm(s, xg.t()).float().cpu().equal(ref.t())                      # sparse first, k contiguous view
    assert torch.mm(s, xg.t().contiguous()).float().cpu().equal(ref.t())         # sparse first, k strided
    assert torch.addmm(bias.to(cuda), xg, s.t()).float().cpu().equal(ref_b)
    out = sparse.sparse_semi_structured_linear(xg, s, bias=bias.to(cuda), activation="relu")
    assert out.float().cpu().equal(ref_b.clamp_min(0))
    # canonical values + metadata through the functional entry point: repacked once, same kernel
    out = sparse.sparse_semi_structured_linear(xg, s.values(), s.indices(), bias=bias.to(cuda))
    assert out.float().cpu().equal(ref_b)


@pytest.mark.parametrize("dims", [(256, 4096, 256), (96, 2048, 520), (352, 12288 // 4, 200)])
def test_spmm_split_k_is_exact_and_deterministic(cuda, dims):
    """k-heavy shapes whose tiles cannot fill the GPU take the split-K path (float32 partial tiles in a
    workspace + reduction launch); small-integer operands keep every partial sum exact."""
    import sparse
    from sparse import _native as N
    n, k, m = dims
    assert N.lib().tf24_spmm_workspace_bytes(N.F16, n, k, m) > 0
    w = _small_ints((n, k), 71, -2, 3).half()
    x = _small_ints((m, k), 72, -2, 3).half()
    bias = _small_ints((n,), 73).half()
    mask = oracle.prune24_mask(w)
    ref = oracle.spmm_ref(x, torch.where(mask, w, torch.zeros_like(w)))
    s = sparse.to_sparse_semi_structured(w.to(cuda))
    out = torch.mm(x.to(cuda), s.t())
    assert out.float().cpu().equal(ref.half().float())
    assert torch.mm(x.to(cuda), s.t()).equal(out)                                  # bit-reproducible
    assert torch.mm(s, x.to(cuda).t().contiguous()).float().cpu().equal(ref.t().half().float())
    outb = torch.addmm(bias.to(cuda), x.to(cuda), s.t())
    assert outb.float().cpu().equal((ref + bias.float()).half().float())


@pytest.mark.parametrize("dtype", [F16, BF16, torch.uint8])
@pytest.mark.parametrize("shape", [(64, 64), (200, 136), (1024, 768), (48, 4096)])
def test_transpose_copy(cuda, dtype, shape):
    from sparse import _native as N
    rows, cols = shape
    if dtype == torch.uint8:
        rows, cols = (rows + 15) // 16 * 16, (cols + 15) // 16 * 16
        t = torch.randint(0, 255, (rows, cols), dtype=torch.uint8, generator=torch.Generator().manual_seed(81))
    else:
        t = randn((rows, cols), dtype, 81)
    out = N.transposed_copy(t.to(cuda))
    assert out.shape == (cols, rows) and out.is_contiguous()
    assert_same(out, t.t().contiguous())


@pytest.mark.parametrize("dtype", [F16, E4M3, torch.int8])
def test_panel_form_is_the_documented_one(cuda, dtype):
    """The panel form as the C header states it, spelled out with torch views of the canonical tensors:
    values [k/KP][m][64 bytes] (KP = 128 / sizeof(value) dense columns), metadata [k/32][m][4 bytes]."""
    import sparse
    from sparse import _native as N
    m, k = 96, 640
    if dtype == torch.int8:
        w = torch.randint(-100, 101, (m, k), generator=torch.Generator().manual_seed(93)).to(torch.int8)
    else:
        w = randn((m, k), F32, 92)
    s = sparse.to_sparse_semi_structured(w.to(cuda), dtype=dtype)
    assert s._store_layout == N.COMPRESSED_PANEL
    want_v, want_m = oracle.compress24(w, out_dtype=dtype)
    kp = 128 // want_v.element_size()
    v_bytes = want_v.contiguous().view(torch.uint8).reshape(m, k // kp, 64).permute(1, 0, 2).contiguous()
    m_bytes = want_m.contiguous().view(torch.uint8).reshape(m, k // 32, 4).permute(1, 0, 2).contiguous()
    assert s._store_values.contiguous().view(torch.uint8).cpu().reshape(k // kp, m, 64).equal(v_bytes)
    assert s._store_meta.contiguous().view(torch.uint8).cpu().reshape(k // 32, m, 4).equal(m_bytes)


@pytest.mark.parametrize("dtype", [F16, E4M3])
def test_repack_between_canonical_and_panel(cuda, dtype):
    """tf24_repack on canonical values/metadata must give the bytes the compress kernel writes in
    panel form, and back."""
    import sparse
    from sparse import _native as N
    m, k = 96, 640
    w = randn((m, k), F32, 91)
    s = sparse.to_sparse_semi_structured(w.to(cuda), dtype=dtype)
    assert s._store_layout == N.COMPRESSED_PANEL
    pv, pm = s._store_values.contiguous(), s._store_meta.contiguous()
    cv, cm = s.values().contiguous(), s.indices().contiguous()
    want_v, want_m = oracle.compress24(w, out_dtype=dtype)
    assert cv.cpu().view(torch.uint8).equal(want_v.view(torch.uint8)) and cm.cpu().equal(want_m)
    ov, om = torch.empty_like(pv), torch.empty_like(pm)
    N.check(N.lib().tf24_repack(cv.data_ptr(), cm.data_ptr(), N.dtype_code(dtype), m, k, N.COMPRESSED_CANONICAL,
                                ov.data_ptr(), om.data_ptr(), N.stream_ptr()))
    assert ov.view(torch.uint8).equal(pv.view(torch.uint8)) and om.view(torch.uint8).equal(pm.view(torch.uint8))
    bv, bm = torch.empty_like(cv), torch.empty_like(cm)
    N.check(N.lib().tf24_repack(pv.data_ptr(), pm.data_ptr(), N.dtype_code(dtype), m, k, N.COMPRESSED_PANEL,
                                bv.data_ptr(), bm.data_ptr(), N.stream_ptr()))
    assert bv.view(torch.uint8).equal(cv.view(torch.uint8)) and bm.view(torch.uint8).equal(cm.view(torch.uint8))
    with pytest.raises(RuntimeError):
        N.check(N.lib().tf24_repack(cv.data_ptr(), cm.data_ptr(), N.dtype_code(dtype), m, k + 8, N.COMPRESSED_CANONICAL,
                                    ov.data_ptr(), om.data_ptr(), N.stream_ptr()))


@pytest.mark.parametrize("dtype,k", [(F16, 64), (F16, 128), (F16, 192), (F16, 256), (BF16, 320), (E4M3, 128), (E4M3, 256), (E5M2, 384)])
def test_spmm_tiled_short_k(cuda, dtype, k):
    """One to five pipeline stages: prologue, steady state and drain of the tiled kernel's stage ring
    each with fewer stages than the ring holds."""
    import sparse
    n, m = 128, 144
    w = _small_ints((n, k), 93).to(dtype)
    x = _small_ints((m, k), 94).to(dtype)
    mask = oracle.prune24_mask(w.float())
    ref = oracle.spmm_ref(x.float(), torch.where(mask, w.float(), torch.zeros(())))
    s = sparse.to_sparse_semi_structured(w.float().to(cuda), dtype=dtype)
    out = torch.mm(x.to(cuda), s.t())
    assert out.float().cpu().equal(ref.to(out.dtype).float())
    out = torch.mm(s, x.to(cuda).t())
    assert out.float().cpu().equal(ref.t().to(out.dtype).float())
    out = torch.mm(s, x.to(cuda).t().contiguous())                                 # k strided: transposing fragment reads
    assert out.float().cpu().equal(ref.t().to(out.dtype).float())


@pytest.mark.parametrize("dtype", [F16, BF16])
def test_spmm_tiled_k_strided_padded_rows(cuda, dtype):
    """`S @ dense` with the dense operand a column slice of a wider row-major matrix: k is the strided
    dimension, rows are longer than the columns used, and the last column tile is partial."""
    import sparse
    n, k, j, ld = 320, 448, 520, 776
    w = _small_ints((n, k), 95).to(dtype)
    wide = _small_ints((k, ld), 96).to(dtype)
    x = wide[:, 8:8 + j]                                                            # [k, j], row pitch ld, 16-byte aligned start
    mask = oracle.prune24_mask(w.float())
    ref = oracle.spmm_ref(x.t().float(), torch.where(mask, w.float(), torch.zeros(()))).t()   # [n, j]
    s = sparse.to_sparse_semi_structured(w.float().to(cuda), dtype=dtype)
    xg = wide.to(cuda)[:, 8:8 + j]
    assert not xg.is_contiguous()
    out = torch.mm(s, xg)
    assert out.float().cpu().equal(ref.to(dtype).float())


# ------------------------------------------------------------------ int8 values and the integer product
def _int8(shape, seed, lo=-128, hi=128):
    return torch.randint(lo, hi, shape, generator=torch.Generator().manual_seed(seed), dtype=torch.int64).to(torch.int8)


@pytest.mark.parametrize("col_major", [False, True])
@pytest.mark.parametrize("use_mask", [False, True])
def test_int8_compress(cuda, col_major, use_mask):
    """int8 dense -> int8 values + int32 metadata (semi_structured.py:24-30, 323-331): magnitude rule
    on |x| with -128 the largest magnitude, ties to the larger index; masks as bytes or floats."""
    import sparse
    w = _int8((96, 384), 101)
    w[:, :8] = torch.tensor([-128, 127, -127, 128 - 256, 5, -5, 5, -5], dtype=torch.int8)   # extremes and ties
    mask = None
    if use_mask:
        _, mask = oracle.transposable_mask(w.float())
        mask[:4] = torch.rand(4, 384, generator=torch.Generator().manual_seed(102)) < 0.5
    want_v, want_m = oracle.compress24(w, mask=mask, out_dtype=torch.int8)
    assert want_v.dtype == torch.int8 and want_m.dtype == torch.int32
    for mk in ([None] if mask is None else [mask, mask.float()]):
        s = sparse.to_sparse_semi_structured(maybe_t(w.to(cuda), col_major),
                                             mask=None if mk is None else maybe_t(mk.to(cuda), col_major), dtype=torch.int8)
        assert s.dtype == torch.int8
        assert_same(s.values(), want_v, "values")
        assert_same(s.indices(), want_m, "meta")
        assert_same(s.to_dense(), oracle.decompress24(want_v, want_m), "to_dense")
    with pytest.raises(RuntimeError):
        sparse.to_sparse_semi_structured(w.to(cuda), dtype=torch.float16)          # int8 tensors give int8 values only
    with pytest.raises(RuntimeError):
        sparse.to_sparse_semi_structured(w.to(cuda).half(), dtype=torch.int8)
    with pytest.raises(RuntimeError):
        sparse.to_sparse_semi_structured(w.to(cuda), dtype=torch.int8, MVUE24=True)


def test_int8_compress_pair(cuda):
    import sparse
    w = _int8((256, 128), 103)
    _, mask = oracle.transposable_mask(w.float())
    want_v, want_m = oracle.compress24(w, mask=mask, out_dtype=torch.int8)
    want_vt, want_mt = oracle.compress24(w.t().contiguous(), mask=mask.t().contiguous(), out_dtype=torch.int8)
    s, s_t = sparse.to_sparse_semi_structured_pair(w.to(cuda), mask.to(cuda), dtype=torch.int8)
    assert_same(s.values(), want_v)
    assert_same(s.indices(), want_m)
    assert_same(s_t.values(), want_vt)
    assert_same(s_t.indices(), want_mt)


@pytest.mark.parametrize("dims", [(32, 128, 16), (64, 256, 40), (352, 640, 304), (256, 4096, 256), (96, 2048, 528)])
def test_int8_spmm_is_exact(cuda, dims):
    """int8 x int8 -> int32 (.cu:594-637) against an int64 product: general kernel, tiled kernel with
    partial tiles, split-K; both operand positions and dense layouts; int32 bias and ReLU."""
    import sparse
    n, k, m = dims
    w, x = _int8((n, k), 111), _int8((m, k), 112)
    bias = torch.randint(-100000, 100000, (n,), generator=torch.Generator().manual_seed(113), dtype=torch.int64).int()
    mask = oracle.prune24_mask(w.float())
    wm = torch.where(mask, w, torch.zeros_like(w))
    ref = oracle.spmm_ref_int(x, wm)
    s = sparse.to_sparse_semi_structured(w.to(cuda), dtype=torch.int8)
    xg = x.to(cuda)
    out = torch.mm(xg, s.t())
    assert out.dtype == torch.int32 and out.cpu().equal(ref)
    assert torch.mm(maybe_t(xg, True), s.t()).cpu().equal(ref)                   # k strided dense operand
    assert torch.mm(s, xg.t()).cpu().equal(ref.t())                              # sparse first
    assert torch.mm(s, xg.t().contiguous()).cpu().equal(ref.t())
    assert torch.addmm(bias.to(cuda), xg, s.t()).cpu().equal(oracle.spmm_ref_int(x, wm, bias))
    out = sparse.sparse_semi_structured_linear(xg, s, bias=bias.to(cuda), activation="relu")
    assert out.cpu().equal(oracle.spmm_ref_int(x, wm, bias, relu=True))
    out = sparse.sparse_semi_structured_linear(xg, s.values(), s.indices())      # canonical pieces
    assert out.cpu().equal(ref)
    with pytest.raises(RuntimeError):
        sparse.sparse_semi_structured_linear(xg, s, activation="silu")           # .cu:610-612: none and ReLU only
    with pytest.raises(RuntimeError):
        torch.mm(xg.half(), s.t())                                               # operand dtypes must match


def test_int8_spmm_extreme_values(cuda):
    """All operands -128: every product is +16384, the sum over k = 2048 kept pairs stays in int32."""
    import sparse
    n, k, m = 64, 4096, 64
    w = torch.full((n, k), -128, dtype=torch.int8)
    x = torch.full((m, k), -128, dtype=torch.int8)
    s = sparse.to_sparse_semi_structured(w.to(cuda), dtype=torch.int8)
    out = torch.mm(x.to(cuda), s.t())
    assert out.cpu().equal(torch.full((m, n), 16384 * (k // 2), dtype=torch.int32))


@pytest.mark.parametrize("dtype,m", [(F16, 8), (BF16, 8), (F16, 24), (BF16, 40), (E4M3, 16), (torch.int8, 16),
                                     (F16, 72), (BF16, 128), (E4M3, 80), (torch.int8, 128)])
@pytest.mark.parametrize("k", [512, 4096])
def test_spmm_narrow_dense_operand(cuda, dtype, m, k):
    """A handful of dense columns against a tall sparse operand: 8 columns take the one-pass kernel,
    up to 64 and up to 128 the tiled kernel on 128 x 64 and 128 x 128 tiles (with k pieces, whose
    partial tiles only cover the live 32-column slabs); every operand position and layout."""
    import sparse
    n = 320
    if dtype == torch.int8:
        w, x = _int8((n, k), 121, -3, 4), _int8((m, k), 122, -3, 4)
        ref = oracle.spmm_ref_int(x, torch.where(oracle.prune24_mask(w.float()), w, torch.zeros_like(w)))
        s = sparse.to_sparse_semi_structured(w.to(cuda), dtype=dtype)
    else:
        w, x = _small_ints((n, k), 121, -2, 3).to(dtype), _small_ints((m, k), 122, -2, 3).to(dtype)
        mask = oracle.prune24_mask(w.float())
        ref = oracle.spmm_ref(x.float(), torch.where(mask, w.float(), torch.zeros(())))
        s = sparse.to_sparse_semi_structured(w.float().to(cuda), dtype=dtype)
    xg = x.to(cuda)
    same = lambda out, want: out.cpu().to(torch.float64).equal(want.to(out.dtype).to(torch.float64))
    assert same(torch.mm(xg, s.t()), ref)
    assert same(torch.mm(maybe_t(xg, True), s.t()), ref)
    assert same(torch.mm(s, xg.t()), ref.t())
    assert same(torch.mm(s, xg.t().contiguous()), ref.t())


@pytest.mark.parametrize("dtype", [F16, E4M3, torch.int8])
@pytest.mark.parametrize("n,k", [(320, 1024), (8192, 1408 * 2)])
def test_spmm_16_columns_without_workspace(cuda, dtype, n, k):
    """Through the C ABI with no workspace the tiled kernel cannot cut k into pieces, and 16 dense
    columns take the one-pass kernel (spmm_few, two waves a row block)."""
    import sparse
    from sparse import _native as N
    m = 16
    if dtype == torch.int8:
        w, x = _int8((n, k), 141, -3, 4), _int8((m, k), 142, -3, 4)
        ref = oracle.spmm_ref_int(x, torch.where(oracle.prune24_mask(w.float()), w, torch.zeros_like(w)))
        s = sparse.to_sparse_semi_structured(w.to(cuda), dtype=dtype)
        out_dtype, out_code = torch.int32, N.I32
    else:
        w, x = _small_ints((n, k), 141, -2, 3).to(dtype), _small_ints((m, k), 142, -2, 3).to(dtype)
        ref = oracle.spmm_ref(x.float(), torch.where(oracle.prune24_mask(w.float()), w.float(), torch.zeros(())))
        s = sparse.to_sparse_semi_structured(w.float().to(cuda), dtype=dtype)
        out_dtype, out_code = torch.float32, N.F32
    xg = x.to(cuda)
    out = torch.empty(m, n, dtype=out_dtype, device=cuda)
    N.check(N.lib().tf24_spmm(s._store_values.data_ptr(), s._store_meta.data_ptr(), N.COMPRESSED_PANEL, N.operand_code(dtype), n, k,
                              xg.data_ptr(), N.ROW_MAJOR, k, m, out.data_ptr(), out_code, N.COL_MAJOR, n, None, 1.0, 0,
                              None, 0, N.stream_ptr()))
    torch.cuda.synchronize()
    assert out.cpu().to(torch.float64).equal(ref.to(torch.float64))


@pytest.mark.parametrize("panels", [1, 17, 22])
@pytest.mark.parametrize("n", [8192, 10272])
@pytest.mark.parametrize("dtype", [F16, E4M3])
def test_spmm_narrow_one_wave_per_block(cuda, dtype, n, panels):
    """Many sparse rows and few dense columns: the one-pass kernel whose blocks own 16 rows, two waves each
    (fewer rows: test_spmm_narrow_dense_operand), with a share of k of no or one panel, of a chunk of eight and a
    panel more, and of one and three more."""
    import sparse
    k, m = panels * (64 if dtype == F16 else 128), 16      # 1 panel, one chunk + 1, 22 panels
    w, x = _small_ints((n, k), 131, -2, 3).to(dtype), _small_ints((m, k), 132, -2, 3).to(dtype)
    mask = oracle.prune24_mask(w.float())
    ref = oracle.spmm_ref(x.float(), torch.where(mask, w.float(), torch.zeros(())))
    s = sparse.to_sparse_semi_structured(w.float().to(cuda), dtype=dtype)
    bias = _small_ints((n,), 133).to(torch.float32 if dtype == E4M3 else dtype)
    out = torch.mm(x.to(cuda), s.t())
    assert out.float().cpu().equal(ref.to(out.dtype).float())
    out = torch.mm(s, x.to(cuda).t())
    assert out.float().cpu().equal(ref.t().to(out.dtype).float())
    out = sparse.sparse_semi_structured_linear(x.to(cuda)[:8], s, bias=bias.to(cuda), activation="relu")
    want = (ref[:8] + bias.float()).clamp_min(0)
    assert out.float().cpu().equal(want.to(out.dtype).float())


def test_narrowing_edge_values(cuda):
    """Float32 -> e4m3 / e5m2 / bf16 / f16 on the device (hardware conversions where gfx950 has them) against
    torch's casts, byte for byte, on the values where narrowing rules differ between implementations:
    the largest finite value and the first one past it (e4m3: 448, ties at 464, NaN from 480 on -- not
    saturation), e5m2's 57344 / 61440 and overflow to infinity, signed infinities and NaNs, signed zeros,
    the subnormal boundaries and halfway cases of each type."""
    import sparse
    edge = [448.0, 449.0, 456.0, 463.99, 464.0, 464.01, 472.0, 479.9, 480.0, 512.0, 1e6, 57344.0, 59000.0, 61439.0, 61440.0, 61441.0,
            65503.0, 65504.0, 65519.9, 65520.0, 65536.0, 1e30, float("inf"), float("nan"), 0.0,
            2.0 ** -6, 2.0 ** -7, 2.0 ** -9, 2.0 ** -10, 1.5 * 2.0 ** -10, 2.0 ** -10 * 1.0001, 2.0 ** -11, 2.0 ** -14, 2.0 ** -16,
            2.0 ** -17, 1.5 * 2.0 ** -17, 2.0 ** -18, 2.0 ** -24, 2.0 ** -25, 1.5 * 2.0 ** -25, 2.0 ** -126, 2.0 ** -133, 2.0 ** -149,
            1.0, 1.0625, 1.09375, 1.125, 1.1875, 3.3895e38, 3.4e38, 240.0, 248.0, 0.0146484375, 0.015625]
    vals = torch.tensor(edge + [-v for v in edge], dtype=torch.float32)
    vals = torch.cat([vals, torch.tensor([0x7fa00001, 0xffc00123 - (1 << 32)], dtype=torch.int32).view(torch.float32)])   # NaNs with payloads
    n = vals.numel()
    k = 128
    rows = (n + 1) // 2 * 4 // k + 1
    rows = (rows + 31) // 32 * 32
    # every value sits at position 0 or 1 of a group whose mask keeps exactly those two positions
    dense = torch.zeros(rows * k, dtype=torch.float32)
    idx = torch.arange(n)
    dense[(idx // 2) * 4 + idx % 2] = vals
    dense = dense.view(rows, k)
    mask = torch.zeros(rows, k, dtype=torch.bool)
    mask.view(-1, 4)[:, :2] = True
    for odt in (E4M3, E5M2, BF16, F16):
        s = sparse.to_sparse_semi_structured(dense.to(cuda), mask=mask.to(cuda), dtype=odt)
        got = s.values().cpu().reshape(-1)[:n]
        want = vals.to(odt)
        gb, wb = got.view(torch.uint8 if odt in FLOAT8 else torch.int16), want.view(torch.uint8 if odt in FLOAT8 else torch.int16)
        nan = vals != vals
        assert gb[~nan].equal(wb[~nan]), (odt, vals[~nan][gb[~nan] != wb[~nan]])
        assert bool((got[nan].float() != got[nan].float()).all()), odt          # NaN stays NaN (payloads are not compared for 16-bit types)
        if odt in FLOAT8:
            assert gb[nan].equal(wb[nan]), odt                                   # one NaN byte per sign, as torch's


@pytest.mark.parametrize("dtype,k,act", [(E4M3, 512, None), (E4M3, 4224, "relu"), (E5M2, 640, "silu"), (F16, 320, "relu"),
                                         (BF16, 2112, None), (torch.int8, 512, None), (torch.int8, 4224, "relu")])
def test_spmm_chained_tiles_32bit_output(cuda, dtype, k, act):
    """More tiles than compute units with a 32-bit output -- float32 from 8-bit operands and int32 from int8, the
    output types the reference gives them (.cu:729, 772; .cu:594-637), float32 from 16-bit ones -- on the chained-tile
    kernel (4 to 5 stages: 8 waves; 33 stages: 4 waves) with its staged 32-bit output pass: 17 x 17 tiles with partial
    edges, bias, activation, against the oracle on exact data, and a second call."""
    import sparse
    n, m = 4128, 4112
    if dtype == torch.int8:
        w, x = _int8((n, k), 121, -20, 21), _int8((m, k), 122, -20, 21)
        bias = torch.randint(-1000, 1000, (n,), generator=torch.Generator().manual_seed(123), dtype=torch.int64).int()
        mask = oracle.prune24_mask(w.float())
        want = oracle.spmm_ref_int(x, torch.where(mask, w, torch.zeros_like(w))) + bias
        if act == "relu":
            want = want.clamp_min(0)
        s = sparse.to_sparse_semi_structured(w.to(cuda), dtype=torch.int8)
        out = sparse.sparse_semi_structured_linear(x.to(cuda), s, bias_opt=bias.to(cuda), activation_opt=act)
        assert out.dtype == torch.int32 and out.shape == (m, n)
        assert out.cpu().equal(want.int())
        assert sparse.sparse_semi_structured_linear(x.to(cuda), s, bias_opt=bias.to(cuda), activation_opt=act).equal(out)
        return
    w = _small_ints((n, k), 124, -2, 3).to(dtype)
    x = _small_ints((m, k), 125, -2, 3).to(dtype)
    bias = _small_ints((n,), 126) * 0.5
    mask = oracle.prune24_mask(w.float())
    pre = oracle.spmm_ref(x.float(), torch.where(mask, w.float(), torch.zeros(()))) * 0.25 + bias
    s = sparse.to_sparse_semi_structured(w.float().to(cuda), dtype=dtype)
    run = lambda: sparse.sparse_semi_structured_linear(x.to(cuda), s, bias_opt=bias.to(cuda), activation_opt=act, out_dtype=torch.float32, scale=0.25)
    out = run()
    assert out.dtype == torch.float32 and out.shape == (m, n)
    got = out.cpu()
    if act in (None, "relu"):
        assert got.equal(pre if act is None else pre.clamp_min(0))
    else:
        want = torch.nn.functional.silu(pre)
        assert bool(((got - want).abs() <= 2e-6 + 2e-6 * want.abs()).all())
    assert run().equal(out)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float8_e4m3fn, torch.int8])
@pytest.mark.parametrize("n,k,rows", [(64, 128, 1), (32, 128, 7), (8192, 256, 3), (10240, 128, 15), (512, 512, 17), (288, 384, 63), (544, 2048, 65),
                                      (768, 256, 127), (256, 4096, 129), (4096, 1024, 255), (3072, 768, 1025), (2304, 4096, 2049), (1600, 6400, 4001)])
def test_linear_any_number_of_rows(cuda, dtype, n, k, rows):
    """tf24_linear against the float32 product on small integers (exact), row counts that are multiples of nothing, on the
    narrow kernels and the 64- and 128-wide tiles; the rows behind the last stay as they were."""
    import sparse
    from sparse import _native as N
    g = torch.Generator().manual_seed(rows)
    w = torch.randint(-2, 3, (n, k), generator=g).float()
    src = w.to(torch.int8) if dtype == torch.int8 else w
    s = sparse.to_sparse_semi_structured(src.to(cuda), dtype=dtype)
    x = torch.randint(-2, 3, (rows, k), generator=g).float().to(cuda)
    out_dtype = torch.int32 if dtype == torch.int8 else torch.float32
    want = (x @ s.to_dense().float().t()).to(out_dtype)
    xs = x.to(dtype)
    y = torch.full((rows + 5, n), 77, dtype=out_dtype, device=cuda)
    code = N.operand_code(dtype)
    ws_bytes = N.lib().tf24_spmm_workspace_bytes(code, n, k, rows)
    ws = torch.empty(max(ws_bytes, 16), dtype=torch.uint8, device=cuda)
    for ws_ptr, ws_len in ((ws.data_ptr(), ws_bytes), (None, 0)):
        y[:rows] = 0
        N.check(N.lib().tf24_linear(s._store_values.data_ptr(), s._store_meta.data_ptr(), N.COMPRESSED_PANEL, code, n, k, xs.data_ptr(), k, rows,
                                    y.data_ptr(), N.operand_code(out_dtype), n, None, 1.0, N.ACT_NONE, ws_ptr, ws_len, N.stream_ptr()))
        assert y[:rows].equal(want)
        assert bool((y[rows:] == 77).all())
    got = torch.mm(xs, s.t())
    assert got.shape == (rows, n) and got.float().equal(want.to(got.dtype).float())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float8_e4m3fn, torch.int8])
@pytest.mark.parametrize("n,stages,rows", [
    (768, 12, 12285),          # 256 x 256 tiles, a workgroup each
    (6144, 192, 757),          # 256 x 256 tiles in three pieces of k
    (4128, 4, 4111),           # 289 tiles on 256 workgroups, chained, eight waves
    (4128, 33, 4111),          # the same, four waves; 256 x 192 tiles with 16-bit results
    (1760, 33, 12271),         # two rounds of 256 x 192 tiles with 16-bit results
    (800, 33, 12271),          # one round of them
    (4128, 33, 8175)])         # full rounds of 256 x 256 tiles, the last tile row in a second launch
def test_linear_ragged_rows_on_wide_tiles(cuda, dtype, n, stages, rows):
    """Row counts that fill no tile on each kernel of more than 256 tiles of 256 x 128, with 32- and 16-bit results; the rows behind
    the last stay as they were.  Exact on small integers.  S @ x.t(), whose results lie the other way round, with the
    rows that are whole multiples of 16."""
    import sparse
    from sparse import _native as N
    k = stages * 128 // torch.empty(0, dtype=dtype).element_size()
    g = torch.Generator(device=cuda).manual_seed(rows + stages)
    w = torch.randint(-2, 3, (n, k), device=cuda, generator=g)
    s = sparse.to_sparse_semi_structured(w.to(torch.int8) if dtype == torch.int8 else w.float(), dtype=dtype)
    x = torch.randint(-2, 3, (rows, k), device=cuda, generator=g).to(dtype)
    want = x.float() @ s.to_dense().float().t()
    code, lib = N.operand_code(dtype), N.lib()
    nbytes = lib.tf24_spmm_workspace_bytes(code, n, k, rows)
    ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=cuda)
    a = (s._store_values.data_ptr(), s._store_meta.data_ptr(), N.COMPRESSED_PANEL, code, n, k, x.data_ptr())
    tail = (None, 1.0, N.ACT_NONE, ws.data_ptr(), nbytes, N.stream_ptr())
    for out_dtype in ((torch.int32,) if dtype == torch.int8 else (torch.float32, torch.float16, torch.bfloat16)):
        y = torch.full((rows + 3, n), 77, dtype=out_dtype, device=cuda)
        N.check(lib.tf24_linear(*a, k, rows, y.data_ptr(), N.operand_code(out_dtype), n, *tail))
        assert y[:rows].equal(want.to(out_dtype)) and bool((y[rows:] == 77).all()), out_dtype
        whole = rows // 16 * 16
        yt = torch.full((n + 1, whole), 77, dtype=out_dtype, device=cuda)
        N.check(lib.tf24_spmm(*a, N.ROW_MAJOR, k, whole, yt.data_ptr(), N.operand_code(out_dtype), N.ROW_MAJOR, whole, *tail))
        assert yt[:n].equal(want[:whole].t().to(out_dtype)) and bool((yt[n] == 77).all()), out_dtype


@pytest.mark.parametrize("dtype,rows,k,view", [
    (torch.float8_e4m3fn, 72, 128, "columns"), (torch.int8, 24, 256, "columns"), (torch.float16, 72, 128, "columns"), (torch.float16, 75, 128, "columns"),
    (torch.float8_e4m3fn, 17, 128, "pitch"), (torch.int8, 88, 128, "pitch"), (torch.bfloat16, 17, 128, "pitch"),
    (torch.float16, 3, 128, "far"), (torch.float8_e4m3fn, 3, 128, "far"), (torch.bfloat16, 1, 128, "far"),
    (torch.bfloat16, 1, 128, "off"), (torch.float16, 17, 128, "off"), (torch.int8, 1, 128, "off"), (torch.float16, 1, 128, "odd"), (torch.float16, 9, 128, "odd")])
@pytest.mark.parametrize("n", [32, 96])
def test_linear_rows_in_views(cuda, dtype, rows, k, view, n):
    """Row counts off the type's multiple in views that the kernels cannot address as they lie: k strided, a pitch of 8 one-byte
    elements, rows more than 16 MiB apart, a start off a
    16-byte boundary, an odd pitch.  Exact: small integers."""
    import sparse
    g = torch.Generator().manual_seed(rows + n)
    w = torch.randint(-2, 3, (n, k), generator=g)
    s = sparse.to_sparse_semi_structured((w if dtype == torch.int8 else w.float()).to(cuda).to(torch.int8 if dtype == torch.int8 else torch.float32), dtype=dtype)
    x = torch.randint(-2, 3, (rows, k), generator=g).float().to(cuda).to(dtype)
    if view == "columns":
        base = torch.zeros(k, rows, dtype=dtype, device=cuda)
        at = base.t()
    elif view == "pitch":
        at = torch.zeros(rows, k + 8, dtype=dtype, device=cuda)[:, :k]
    elif view == "off":
        at = torch.zeros(rows * k + 1, dtype=dtype, device=cuda)[1:].view(rows, k)
    elif view == "odd":
        at = torch.zeros(rows, k + 1, dtype=dtype, device=cuda)[:, :k]
    else:
        at = torch.zeros(rows, (1 << 24) // x.element_size() + 16, dtype=dtype, device=cuda)[:, :k]
    at.copy_(x)
    want = x.float() @ s.to_dense().float().t()
    for got in (torch.mm(at, s.t()), sparse.sparse_semi_structured_linear(at, s)):
        assert got.shape == (rows, n) and got.float().equal(want.to(got.dtype).float())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float8_e4m3fn, torch.int8])
@pytest.mark.parametrize("n,panels", [(32, 1), (256, 5), (4096, 24), (4128, 24), (4096, 25), (768, 32), (4096, 33), (96, 64), (6144, 9), (8192, 17), (8224, 3), (4128, 33), (7168, 64),
                                      (4128, 65), (8192, 33), (12288, 16), (12320, 5), (10240, 17)])
def test_few_dense_columns(cuda, dtype, n, panels):
    """Dense extents up to and past those that the narrow kernels take, both output orders; exact on small integers."""
    import sparse
    from sparse import _native as N
    k = panels * 128 // torch.empty(0, dtype=dtype).element_size()
    g = torch.Generator(device=cuda).manual_seed(n + panels)
    w = torch.randint(-2, 3, (n, k), device=cuda, generator=g)
    s = sparse.to_sparse_semi_structured(w.to(torch.int8) if dtype == torch.int8 else w.float(), dtype=dtype)
    dense = s.to_dense().float()
    out_dtype = torch.int32 if dtype == torch.int8 else torch.float32
    code = N.operand_code(dtype)
    bias = torch.randint(-5, 6, (n,), device=cuda, generator=g).to(out_dtype)
    for rows in (8, 9, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65):
        x = torch.randint(-2, 3, (rows, k), device=cuda, generator=g).to(dtype)
        want = (x.float() @ dense.t() + bias.float()).to(out_dtype)
        nbytes = N.lib().tf24_spmm_workspace_bytes(code, n, k, rows)
        ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=cuda)
        y = torch.full((rows + 1, n), 77, dtype=out_dtype, device=cuda)
        N.check(N.lib().tf24_linear(s._store_values.data_ptr(), s._store_meta.data_ptr(), N.COMPRESSED_PANEL, code, n, k, x.data_ptr(), k, rows, y.data_ptr(),
                                    N.operand_code(out_dtype), n, bias.data_ptr(), 1.0, N.ACT_NONE, ws.data_ptr(), nbytes, N.stream_ptr()))
        assert y[:rows].equal(want) and bool((y[rows:] == 77).all()), rows
        if rows % 16 == 0:
            yt = torch.full((n, rows), 77, dtype=out_dtype, device=cuda)
            N.check(N.lib().tf24_spmm(s._store_values.data_ptr(), s._store_meta.data_ptr(), N.COMPRESSED_PANEL, code, n, k, x.data_ptr(), N.ROW_MAJOR, k, rows,
                                      yt.data_ptr(), N.operand_code(out_dtype), N.ROW_MAJOR, rows, bias.data_ptr(), 1.0, N.ACT_NONE, ws.data_ptr(), nbytes,
                                      N.stream_ptr()))
            assert yt.equal(want.t()), rows


@pytest.mark.parametrize("dtype", [torch.float16, torch.float8_e4m3fn])
@pytest.mark.parametrize("n,panels", [(96, 11), (416, 12), (4096, 23), (4128, 23),            # two waves a row block, a share of five panels and more
                                      (1056, 25), (6144, 49), (8160, 31),                     # four
                                      (32, 48), (1568, 49), (4096, 131), (1536, 191),         # eight, shares of one chunk and of several, odd ones
                                      (8192, 129), (10272, 18)])                              # two again
def test_one_to_thirty_two_rows(cuda, dtype, n, panels):
    """Few rows against a weight whose row blocks are shared by two, four and eight waves, in whole and partial chunks of panels: exact
    on small integers, the row behind the last stays as it was."""
    import sparse
    from sparse import _native as N
    k = panels * 128 // torch.empty(0, dtype=dtype).element_size()
    g = torch.Generator(device=cuda).manual_seed(n + panels)
    s = sparse.to_sparse_semi_structured(torch.randint(-2, 3, (n, k), device=cuda, generator=g).float(), dtype=dtype)
    dense = s.to_dense().float()
    for rows in (1, 2, 3, 7, 8, 9, 10, 15, 16, 17, 24, 25, 31, 32):
        x = torch.randint(-2, 3, (rows, k), device=cuda, generator=g).to(dtype)
        y = torch.full((rows + 1, n), 77, dtype=torch.float32, device=cuda)
        N.check(N.lib().tf24_linear(s._store_values.data_ptr(), s._store_meta.data_ptr(), N.COMPRESSED_PANEL, N.operand_code(dtype), n, k, x.data_ptr(), k, rows,
                                    y.data_ptr(), N.F32, n, None, 1.0, N.ACT_NONE, None, 0, N.stream_ptr()))
        assert y[:rows].equal(x.float() @ dense.t()) and bool((y[rows:] == 77).all()), rows


SMALL_TILES = [(64, 1, 65), (96, 2, 127), (128, 3, 128), (160, 4, 129), (288, 5, 200), (32 * 35, 6, 255), (992, 7, 1000), (640, 8, 4001),
               (1024, 12, 300), (4096, 28, 72), (2080, 27, 1900),                                # one piece of k: around the four stage buffers, and long
               (96, 29, 66), (1184, 30, 136), (672, 64, 520), (160, 77, 1345), (1600, 100, 250)]    # pieces
LOWER_TILES = [(320, 20, 11001), (960, 21, 4208), (992, 23, 4297), (4128, 22, 1001), (11008, 20, 304), (1184, 40, 3584), (2048, 176, 2176)]    # 192 x 128
MID_TILES = [(4128, 5, 1104), (320, 19, 11001)]                                                  # 256 x 128
SLIM_TILES = [(4128, 1, 33), (8224, 2, 17), (8224, 3, 64), (5120, 4, 49), (8224, 5, 24), (8224, 6, 32), (8224, 7, 63), (96, 25, 49), (160, 28, 40),    # 128 x 64, whole
              (96, 29, 64), (1184, 67, 24), (672, 100, 33), (160, 77, 17), (64, 129, 16),          # in pieces
              (16416, 64, 40), (16416, 66, 63)]                                                        # whole, where only 256 x 64 tiles could be cut


@pytest.mark.parametrize("dtype", [torch.float16, torch.float8_e4m3fn, torch.int8])
@pytest.mark.parametrize("n,stages,rows", SMALL_TILES + LOWER_TILES + MID_TILES + SLIM_TILES)
def test_tiles_of_64_and_128_columns(cuda, dtype, n, stages, rows):
    """Rows and columns that do not fill their last tile, one stage and more, whole and in pieces, either order of the results, with bias
    and without: exact on small integers, the row behind the last stays as it was."""
    import sparse
    from sparse import _native as N
    k = stages * 128 // torch.empty(0, dtype=dtype).element_size()
    code, wide = N.operand_code(dtype), torch.int32 if dtype == torch.int8 else torch.float32
    g = torch.Generator(device=cuda).manual_seed(n + stages + rows)
    s = sparse.to_sparse_semi_structured(torch.randint(-2, 3, (n, k), device=cuda, generator=g).to(torch.int8 if dtype == torch.int8 else torch.float32), dtype=dtype)
    x = torch.randint(-2, 3, (rows, k), device=cuda, generator=g).to(dtype)
    want = x.float() @ s.to_dense().float().t()                   # (whole numbers below 2**24)
    ws = torch.empty(max(N.lib().tf24_spmm_workspace_bytes(code, n, k, rows), 16), dtype=torch.uint8, device=cuda)
    for out_dtype in (wide,) if dtype == torch.int8 else (wide, torch.float16):
        bias = torch.randint(-4, 5, (n,), device=cuda, generator=g).to(out_dtype)
        for b in (None, bias):
            y = torch.full((rows + 1, n), 77, dtype=out_dtype, device=cuda)
            N.check(N.lib().tf24_linear(s._store_values.data_ptr(), s._store_meta.data_ptr(), N.COMPRESSED_PANEL, code, n, k, x.data_ptr(), k, rows, y.data_ptr(),
                                        N.operand_code(out_dtype), n, None if b is None else b.data_ptr(), 1.0, N.ACT_NONE, ws.data_ptr(), ws.numel(), N.stream_ptr()))
            assert y[:rows].equal((want + (0 if b is None else b.float())).to(out_dtype)) and bool((y[rows:] == 77).all()), (out_dtype, b is None)
    for out_dtype in ((wide, torch.float16)[:1 + (dtype != torch.int8)] if rows % (8 if dtype == torch.float16 else 16) == 0 else ()):
        yt = torch.full((n, rows), 77, dtype=out_dtype, device=cuda)
        N.check(N.lib().tf24_spmm(s._store_values.data_ptr(), s._store_meta.data_ptr(), N.COMPRESSED_PANEL, code, n, k, x.data_ptr(), N.ROW_MAJOR, k, rows,
                                  yt.data_ptr(), N.operand_code(out_dtype), N.ROW_MAJOR, rows, None, 1.0, N.ACT_NONE, ws.data_ptr(), ws.numel(), N.stream_ptr()))
        assert yt.equal(want.t().to(out_dtype)), out_dtype


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float8_e4m3fn, torch.int8])
@pytest.mark.parametrize("n,stages,rows", [(64, 1, 65), (160, 4, 129), (1184, 30, 136), (672, 64, 520), (2080, 27, 1900),          # 128 x 128 tiles, whole and in pieces
                                           (320, 20, 11001), (1184, 40, 3584),                                                  # 192 x 128
                                           (8224, 3, 64), (96, 25, 49), (160, 28, 40), (672, 100, 33)])                         # 128 x 64
def test_tiles_of_64_and_128_columns_with_activation(cuda, dtype, n, stages, rows):
    """The kernels with an activation, a bias in the results' type and in float32, and as much scratch as asked for, half of it (fewer
    pieces) and none: exact on small integers, the row behind the last stays as it was."""
    import sparse
    from sparse import _native as N
    k = stages * 128 // torch.empty(0, dtype=dtype).element_size()
    code, out_dtype = N.operand_code(dtype), torch.int32 if dtype == torch.int8 else torch.float16 if dtype == torch.float8_e4m3fn else dtype
    g = torch.Generator(device=cuda).manual_seed(n + stages + rows)
    s = sparse.to_sparse_semi_structured(torch.randint(-2, 3, (n, k), device=cuda, generator=g).to(torch.int8 if dtype == torch.int8 else torch.float32), dtype=dtype)
    x = torch.randint(-2, 3, (rows, k), device=cuda, generator=g).to(dtype)
    bias = torch.randint(-4, 5, (n,), device=cuda, generator=g)
    want = (x.float() @ s.to_dense().float().t() + bias).clamp_min(0).to(out_dtype)                  # (whole numbers below 2**24)
    asked = N.lib().tf24_spmm_workspace_bytes(code, n, k, rows)
    ws = torch.empty(max(asked, 16), dtype=torch.uint8, device=cuda)
    for b, flag in [(bias.to(out_dtype), 0)] + ([(bias.float(), N.BIAS_F32)] if out_dtype != torch.int32 else []):
        for scratch in {asked, asked // 2 // 16 * 16, 0}:
            y = torch.full((rows + 1, n), 77, dtype=out_dtype, device=cuda)
            N.check(N.lib().tf24_linear(s._store_values.data_ptr(), s._store_meta.data_ptr(), N.COMPRESSED_PANEL, code, n, k, x.data_ptr(), k, rows, y.data_ptr(),
                                        N.operand_code(out_dtype), n, b.data_ptr(), 1.0, N.ACT_RELU | flag, ws.data_ptr() if scratch else None, scratch, N.stream_ptr()))
            assert y[:rows].equal(want) and bool((y[rows:] == 77).all()), (flag, scratch)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float8_e4m3fn])
@pytest.mark.parametrize("n,panels", [(4096, 64), (4096, 65), (512, 32), (512, 33), (6144, 32), (8192, 16), (8192, 17)])      # shares of whole chunks (8 panels, 4 from 17 rows on), and one panel more
def test_one_to_thirty_two_rows_at_the_edges_of_chunks(cuda, dtype, n, panels):
    test_one_to_thirty_two_rows(cuda, dtype, n, panels)


TALL_SLIM_TILES = [(16416, 102, 40), (17440, 133, 63), (32800, 12, 33), (33056, 13, 64)]       # 256 x 64, in pieces and whole (test_launches.py)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float8_e4m3fn, torch.int8])
@pytest.mark.parametrize("n,stages,rows", TALL_SLIM_TILES + [(98336, 1, 17), (16416, 101, 64)])
def test_tiles_of_64_columns_of_tall_weights(cuda, dtype, n, stages, rows):
    test_tiles_of_64_and_128_columns(cuda, dtype, n, stages, rows)


MID_PIECES = [(1600, 100, 1297), (4096, 86, 457), (1280, 80, 1432)]       # 256 x 128, in pieces (test_launches.py)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float8_e4m3fn, torch.int8])
@pytest.mark.parametrize("n,stages,rows", MID_PIECES)
def test_tiles_of_128_columns_in_pieces(cuda, dtype, n, stages, rows):
    test_tiles_of_64_and_128_columns(cuda, dtype, n, stages, rows)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float8_e4m3fn])
@pytest.mark.parametrize("n,panels", [(32, 1), (256, 4), (2144, 5), (4096, 7), (4128, 7), (8192, 7), (8224, 7), (4096, 8)])
def test_one_to_thirty_two_rows_of_a_short_k(cuda, dtype, n, panels):
    test_one_to_thirty_two_rows(cuda, dtype, n, panels)


@pytest.mark.parametrize("dtype,special", [(F16, float("inf")), (BF16, float("-inf")), (E5M2, float("inf")), (E4M3, float("nan"))])
@pytest.mark.parametrize("n,panels", [(768, 12), (512, 11), (256, 5), (4096, 22), (1024, 37), (8192, 17), (8224, 3), (10240, 43)])
def test_few_dense_columns_special_values(cuda, dtype, special, n, panels):
    """An infinity or NaN among the activations reaches only the outputs whose weight keeps its position, as itself, also in
    the last panel, where a batch of panels may end early.  All kept weights are non-zero integers: exact."""
    import sparse
    width = 128 // torch.empty(0, dtype=dtype).element_size()
    k = panels * width
    g = torch.Generator(device=cuda).manual_seed(n + panels)
    w = torch.randint(1, 3, (n, k), device=cuda, generator=g).float() * (torch.randint(0, 2, (n, k), device=cuda, generator=g) * 2 - 1).float()
    s = sparse.to_sparse_semi_structured(w, dtype=dtype)
    dense = s.to_dense().float()
    for rows in (1, 8, 13, 16, 29, 45, 64):
        x = torch.randint(-2, 3, (rows, k), device=cuda, generator=g).float()
        at = torch.tensor([(k - 3, k - width, 0, k - 9)[r % 4] for r in range(rows)], device=cuda)      # row r is special in column at[r]
        line = torch.arange(rows, device=cuda)
        x[line, at] = 0
        want = x @ dense.t()
        hit = dense.t()[at]                                                                           # [rows, n]: the weights it meets
        want = torch.where(hit != 0, special * hit, want)
        x[line, at] = special
        got = torch.mm(x.to(dtype), s.t())
        assert torch.allclose(got.float(), want.to(got.dtype).float(), rtol=0, atol=0, equal_nan=True), rows


@pytest.mark.parametrize("dtype,pitch", [(F16, 0), (BF16, 0), (E4M3, 0), (E4M3, 8), (torch.int8, 8)])
@pytest.mark.parametrize("rows", [8, 16, 48])
@pytest.mark.parametrize("view", ["far", "off"])
def test_products_of_views_at_full_multiples(cuda, dtype, pitch, rows, view):
    """Row counts that are multiples of everything, in views that start off a 16-byte boundary, whose rows are more than 16 MiB
    apart or have a pitch of 8 one-byte elements: the rows of x @ S.t() and of S @ x.t(), where an odd count works too.
    Exact: small integers."""
    import sparse
    k = 128
    g = torch.Generator().manual_seed(rows)
    w = torch.randint(-2, 3, (64, k), generator=g)
    s = sparse.to_sparse_semi_structured((w.to(torch.int8) if dtype == torch.int8 else w.float()).to(cuda), dtype=dtype)
    x = torch.randint(-2, 3, (rows, k), generator=g).float().to(cuda).to(dtype)
    if view == "off":
        at = torch.zeros(rows * (k + pitch) + 1, dtype=dtype, device=cuda)[1:].view(rows, k + pitch)[:, :k]
    elif pitch:
        at = torch.zeros(rows, k + pitch, dtype=dtype, device=cuda)[:, :k]
    else:
        at = torch.zeros(rows, (1 << 24) // x.element_size() + 16, dtype=dtype, device=cuda)[:, :k]
    at.copy_(x)
    want = x.float() @ s.to_dense().float().t()
    for got in (torch.mm(at, s.t()), sparse.sparse_semi_structured_linear(at, s), torch.mm(s, at.t()).t()):
        assert got.shape == (rows, 64) and got.float().equal(want.to(got.dtype).float())


# rows of the weight, stages of 128 bytes of k, dense rows; the tiles that products with 16-bit results take, and whether their
# stages start at another eighth of k on each XCD (test_tile_rules.py holds both against the rules)
STAGE_ORDER = [
    (4384, 55, 5766, "wide", False),                # every XCD from the first stage on
    (4384, 56, 5766, "wide", True),                 # from here on each from its own eighth of k
    (4384, 59, 5766, "wide", True),                 # eighths of unequal length
    (4960, 59, 6428, "wide, two launches", True),   # full rounds of 256 x 256 tiles, the last tile row on others
    (800, 59, 12271, "narrow", True),               # one round of 256 x 192 tiles
    (1568, 66, 10814, "narrow", True),              # two of them
    (4128, 59, 4111, "square", True),               # 192 x 192 tiles, partial ones on either edge
    (3040, 56, 6130, "square", True)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float8_e4m3fn, torch.int8])
@pytest.mark.parametrize("n,stages,rows", [case[:3] for case in STAGE_ORDER])
def test_linear_stage_order_by_xcd(cuda, dtype, n, stages, rows):
    """Long tiles whose stages start at another eighth of k on each XCD and wrap round: exact on small integers, with
    32- and 16-bit results (256 x 256, 256 x 192 and 192 x 192 tiles), and the same again on a second call."""
    import sparse
    k = stages * 128 // torch.empty(0, dtype=dtype).element_size()
    g = torch.Generator(device=cuda).manual_seed(rows + stages)
    w = torch.randint(-2, 3, (n, k), device=cuda, generator=g)
    s = sparse.to_sparse_semi_structured(w.to(torch.int8) if dtype == torch.int8 else w.float(), dtype=dtype)
    x = torch.randint(-2, 3, (rows, k), device=cuda, generator=g).to(dtype)
    want = x.float() @ s.to_dense().float().t()
    for out_dtype in {torch.int8: (torch.int32,)}.get(dtype, (torch.float32, dtype if dtype.itemsize == 2 else torch.bfloat16)):
        got = sparse.sparse_semi_structured_linear(x, s, out_dtype=out_dtype)
        assert got.equal(want.to(out_dtype))
        assert sparse.sparse_semi_structured_linear(x, s, out_dtype=out_dtype).equal(got)


SQUARE = [
    (736, 4, 12271, False),         # one round, the shortest tiles; partial ones on either edge
    (768, 5, 12288, False),         # 256 full tiles
    (3040, 5, 6130, False),         # two rounds, every second workgroup starts late
    (3040, 33, 6130, False),        # the same, together
    (3040, 67, 6130, True)]         # from another eighth of k on each XCD


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("n,stages,rows", [case[:3] for case in SQUARE])
@pytest.mark.parametrize("activation", [None, "relu"])
def test_linear_square_tiles(cuda, dtype, n, stages, rows, activation):
    """Products on 192 x 192 tiles, with and without bias: exact on small integers."""
    import sparse
    k = stages * 128 // torch.empty(0, dtype=dtype).element_size()
    g = torch.Generator(device=cuda).manual_seed(rows + stages)
    s = sparse.to_sparse_semi_structured(torch.randint(-1, 2, (n, k), device=cuda, generator=g).float(), dtype=dtype)
    x = torch.randint(-1, 2, (rows, k), device=cuda, generator=g).to(dtype)
    out_dtype = torch.bfloat16 if dtype == torch.float8_e4m3fn else dtype
    bias = torch.randint(-3, 4, (n,), device=cuda, generator=g).to(out_dtype)
    want = x.float() @ s.to_dense().float().t()
    act = torch.relu if activation else (lambda t: t)
    assert sparse.sparse_semi_structured_linear(x, s, out_dtype=out_dtype, activation=activation).equal(act(want).to(out_dtype))
    assert sparse.sparse_semi_structured_linear(x, s, bias=bias, out_dtype=out_dtype, activation=activation).equal(act(want + bias.float()).to(out_dtype))


TALL = [
    (1504, 24, 11707, False),       # one round, the fewest stages; partial tiles on either edge
    (1120, 44, 14480, False),       # the last of three tile rows reaches 32 rows past its first wave
    (3872, 45, 8535, False),        # two rounds
    (2912, 58, 12074, True)]        # from another eighth of k on each XCD
NOT_TALL = [                        # on the tiles of the cases above that 16-bit operands leave for tall ones
    (1568, 33, 9867, "square"), (1568, 66, 9867, "square"), (3104, 59, 10790, "wide, two launches")]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,stages,rows", [case[:3] for case in TALL + NOT_TALL])
@pytest.mark.parametrize("activation", [None, "relu"])
def test_linear_tall_tiles(cuda, dtype, n, stages, rows, activation):
    """Products on 384 x 192 tiles, with and without bias: exact on small integers."""
    test_linear_square_tiles(cuda, dtype, n, stages, rows, activation)


SHORT = [                           # fewer stages than chained 256 x 256 tiles take on four waves: (form on 16-bit operands, on 8-bit ones)
    (2080, 4, 10541, "narrow", "narrow"),               # the fewest stages; two rounds, partial tiles on either edge
    (3072, 12, 12288, "narrow", "narrow"),              # three full rounds
    (800, 12, 10188, "narrow", "narrow"),               # one round, the fewest stages for that
    (640, 31, 12472, "narrow", "narrow"),               # the most stages
    (1312, 8, 11029, "tall", "square"),                 # the fewest stages of tall tiles
    (3456, 12, 10590, "tall", "wide"), (1120, 31, 12811, "tall", "wide")]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("n,stages,rows", [case[:3] for case in SHORT])
@pytest.mark.parametrize("activation", [None, "relu"])
def test_linear_narrow_and_tall_tiles_of_few_stages(cuda, dtype, n, stages, rows, activation):
    """Products on chained 256 x 192 and 384 x 192 tiles of few stages, with and without bias: exact on small integers."""
    test_linear_square_tiles(cuda, dtype, n, stages, rows, activation)


SQUARE_STRIDED = [                  # and in how many pieces of k (test_tile_rules.py)
    (64, 4, 72, 1), (224, 5, 200, 1), (192, 9, 192, 3), (352, 25, 2376, 3), (416, 8, 560, 1),         # tiles past either edge
    (992, 40, 392, 5), (544, 117, 120, 15), (3072, 48, 768, 2), (3424, 202, 80, 11)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,stages,cols", [case[:3] for case in SQUARE_STRIDED])
def test_spmm_square_tiles_k_strided(cuda, dtype, n, stages, cols):
    """Products with a k-strided dense operand on 192 x 192 tiles, in one and in several pieces: exact on small integers, with
    float32 and 16-bit results of either order."""
    import sparse
    from sparse.semi_structured import _spmm
    k = stages * 64
    g = torch.Generator(device=cuda).manual_seed(n + stages)
    s = sparse.to_sparse_semi_structured(torch.randint(-1, 2, (n, k), device=cuda, generator=g).float(), dtype=dtype)
    x = torch.randint(-1, 2, (k, cols), device=cuda, generator=g).to(dtype)
    want = s.to_dense().float() @ x.float()
    assert _spmm(s, x, True, out_dtype=torch.float32).equal(want)
    assert torch.mm(s, x).equal(want.to(dtype))
    assert torch.mm(x.t(), s.t()).equal(want.t().to(dtype))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k,rows", [(32, 64, 5), (256, 256, 3), (8192, 128, 7), (4096, 4096, 40), (1024, 4096, 100),      # general, narrow, slim, half tiles
                                      (6144, 192 * 64, 757), (4128, 192, 4111), (4128, 2112, 4111), (3040, 320, 6130)])     # pieces, 256 x 256, 192 x 192
@pytest.mark.parametrize("activation", [None, "relu"])
def test_linear_float32_bias_is_rounded(cuda, dtype, n, k, rows, activation):
    """A float32 bias with 16-bit results: the same bits as the bias rounded by the caller, in every kernel."""
    import sparse
    g = torch.Generator(device=cuda).manual_seed(n + rows)
    s = sparse.to_sparse_semi_structured(torch.randn(n, k, device=cuda, generator=g), dtype=dtype)
    x = torch.randn(rows, k, device=cuda, generator=g).to(dtype)
    bias = 3 * torch.randn(n, device=cuda, generator=g)
    bias[::7] *= 1e-6                                              # (subnormal in half precision)
    call = lambda b: sparse.sparse_semi_structured_linear(x, s, bias=b, activation=activation)
    assert call(bias).equal(call(bias.to(dtype)))
    for b in (bias, bias.to(dtype)):
        assert call(torch._neg_view(b)).equal(call(-b))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,k", [(1, 4), (8, 8), (300, 1028)])
def test_soft_threshold_scaled_with_bias(cuda, dtype, m, k):
    from sparse import _native as N
    g = torch.Generator(device=cuda).manual_seed(m)
    w, b = torch.randn(m, k, device=cuda, generator=g), torch.randn(m, device=cuda, generator=g)
    want, out, rounded = (torch.empty(shape, dtype=dtype, device=cuda) for shape in ((m, k), (m, k), (m,)))
    code = N.dtype_code(dtype)
    N.check(N.lib().tf24_soft_threshold24_scaled(w.data_ptr(), m, k, None, 1.25, want.data_ptr(), code, N.stream_ptr()))
    N.check(N.lib().tf24_soft_threshold24_scaled_bias(w.data_ptr(), m, k, None, 1.25, out.data_ptr(), b.data_ptr(), rounded.data_ptr(), code, N.stream_ptr()))
    assert out.equal(want) and rounded.equal(b.to(dtype))
