"""GPU integration: SparseLinearTranspose forward/backward against a dense masked autograd model,
a short masked-decay training loop (reduced), and the fp8 path of config 5."""
import pytest
import torch
import torch.nn.functional as F

import oracle

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.float() - b.float()).norm() / b.float().norm()).item()


def test_sparse_linear_transpose_matches_dense_masked(cuda):
    import sparse
    torch.manual_seed(0)
    layer = sparse.SparseLinearTranspose(256, 512, bias=True).to(cuda)
    x = torch.randn(4, 64, 256, device=cuda, requires_grad=True)
    y = layer(x)
    assert y.shape == (4, 64, 512) and y.dtype == torch.float16
    w = layer.weight.detach()
    # the mask is the transposable one of the master weight (bit-exact with the oracle)
    _, want_mask = oracle.transposable_mask(w.float().cpu())
    assert layer.weight.mask.cpu().equal(want_mask)
    wm = (w * layer.weight.mask).half()
    y_ref = F.linear(x.detach().half(), wm, layer.bias.detach().half())
    assert _rel(y, y_ref) < 1e-2
    gy = torch.randn_like(y)
    y.backward(gy)
    dx_ref = gy.reshape(-1, 512).float() @ wm.float()
    assert _rel(x.grad.reshape(-1, 256), dx_ref) < 1e-2
    db_ref = gy.reshape(-1, 512).float().sum(0)
    assert _rel(layer.bias.grad, db_ref) < 1e-2
    # dW is an MVUE estimate of dY^T x (pruned along the token axis): unbiased, so the mean of
    # several draws converges to the dense gradient
    dw_ref = gy.reshape(-1, 512).float().t() @ x.detach().reshape(-1, 256).half().float()
    assert layer.weight.grad.shape == (512, 256)
    single = _rel(layer.weight.grad, dw_ref)
    draws = []
    for _ in range(24):
        layer.weight.grad = None
        layer.weight.cnt = 0
        x2 = x.detach().clone().requires_grad_(True)
        layer(x2).backward(gy)
        draws.append(layer.weight.grad.float())
    mean_err = _rel(torch.stack(draws).mean(0), dw_ref)
    assert single < 1.0 and mean_err < 0.25 and mean_err < 0.6 * single, (single, mean_err)


def test_layer_state_machine(cuda):
    import sparse
    torch.manual_seed(1)
    layer = sparse.SparseLinearTranspose(128, 128, bias=False).to(cuda)
    w = layer.weight
    assert (w.freq, w.cnt, w.counter, w.step, w.mode) == (40, 0, 0, 0, 'sparse')
    x = torch.randn(32, 128, device=cuda)
    layer(x)
    first = w.weight_sparse
    assert (w.cnt, w.counter, w.step) == (1, 1, 1)
    layer(x)                                     # gradient accumulation: no recompression
    assert w.weight_sparse is first and (w.cnt, w.counter, w.step) == (2, 1, 2)
    w.cnt = 0                                    # what the optimizer hook does
    layer(x)
    assert w.weight_sparse is not first and w.counter == 2
    w.mode = 'dense'
    y = layer(x)
    assert torch.allclose(y, F.linear(x, w), atol=1e-5)
    layer.eval()
    w.mode = 'sparse'
    before = (w.cnt, w.counter, w.step)
    layer(x)
    assert (w.cnt, w.counter, w.step) == before


def test_masked_decay_training_loop(cuda):
    """BASELINE config 4 at reduced size: GELU MLP of two SparseLinearTranspose layers, fused
    AdamW, masked decay alpha = 2e-4 before every optimizer step, mask refresh every 5 steps."""
    import sparse
    torch.manual_seed(2)
    tokens, d, h = 512, 128, 256
    fc, proj = sparse.SparseLinearTranspose(d, h).to(cuda), sparse.SparseLinearTranspose(h, d).to(cuda)
    for layer in (fc, proj):
        torch.nn.init.normal_(layer.weight, std=0.02)
        layer.weight.freq = 5
    params = list(fc.parameters()) + list(proj.parameters())
    opt = torch.optim.AdamW(params, lr=3e-3, weight_decay=0.0, fused=True)
    x = torch.randn(tokens, d, device=cuda)
    target = torch.tanh(x @ torch.randn(d, d, device=cuda) * 0.3)
    losses, masks = [], []
    for step in range(20):
        out = proj(F.gelu(fc(x)))
        loss = F.mse_loss(out.float(), target)
        opt.zero_grad(set_to_none=True)
        loss.backward()
        with torch.no_grad():
            for p in params:
                if hasattr(p, 'mask') and p.mode == 'sparse':
                    p.grad = p.grad.float()
                    before = p.grad.clone()
                    sparse.masked_add_(p.grad.data, p.data, p.mask, alpha=2e-4)
                    want = oracle.masked_add(before.cpu(), p.data.cpu(), p.mask.cpu(), alpha=2e-4)
                    assert p.grad.cpu().equal(want)
                    p.cnt = 0
        opt.step()
        losses.append(loss.item())
        masks.append(fc.weight.mask.clone())
        if step % 5 == 0:       # refreshed on this forward pass from the weights before the update
            blk = fc.weight.mask.reshape(h // 4, 4, d // 4, 4)
            assert blk.sum(1).eq(2).all() and blk.sum(3).eq(2).all()
    assert losses[-1] < 0.7 * losses[0], losses
    assert masks[1].equal(masks[4]) and fc.weight.counter == 20       # constant between refreshes
    assert all(torch.isfinite(torch.tensor(losses)))


def test_fp8_mvue_spmm_config5_reduced(cuda):
    """Config 5 at reduced size: per-tensor amax scaling to e4m3, B pruned by MVUE24 with seeded
    uniforms, fp8 SMFMAC product with bf16 output, against the dense fp32 masked product."""
    import sparse
    g = torch.Generator().manual_seed(5)
    A = torch.randn(512, 1024, generator=g)
    B = torch.randn(256, 1024, generator=g)
    U = torch.rand(256, 1024, generator=g)
    sa, sb = 448.0 / A.abs().max(), 224.0 / B.abs().max()        # headroom: MVUE rescales kept values by up to 2x+
    Aq = (A * sa).to(torch.float8_e4m3fn)
    Bs = (B * sb).bfloat16()
    want_v, want_m, mask = oracle.mvue24(Bs, U, out_dtype=torch.float8_e4m3fn)
    s = sparse.to_sparse_semi_structured(Bs.to(cuda), MVUE24=True, rand=U.to(cuda), dtype=torch.float8_e4m3fn)
    assert s.values().cpu().view(torch.uint8).equal(want_v.view(torch.uint8))
    assert s.indices().cpu().equal(want_m)
    dense_b = oracle.decompress24(want_v, want_m).float()
    ref = (Aq.float() @ dense_b.t()) / (sa * sb)
    out = sparse.sparse_semi_structured_linear(Aq.to(cuda), s, out_dtype=torch.bfloat16, scale=float(1.0 / (sa * sb)))
    assert out.dtype == torch.bfloat16 and out.shape == (512, 256)
    assert _rel(out.cpu(), ref) < 5e-2
    # default dispatch returns float32 like the reference's CUTLASS path
    out32 = torch.mm(Aq.to(cuda), s.t())
    assert out32.dtype == torch.float32 and _rel(out32.cpu() / (sa * sb), ref) < 5e-2
    # soft threshold on the bf16 operand, as config 5 applies every iteration
    sp, mk = sparse.soft_threshold24_triton(Bs.to(cuda))
    wsp, wmk = oracle.soft_threshold24(Bs)
    assert sp.cpu().view(torch.int16).equal(wsp.view(torch.int16)) and mk.cpu().view(torch.int16).equal(wmk.view(torch.int16))


def test_functional_linear_entry_point(cuda):
    import sparse
    g = torch.Generator().manual_seed(6)
    w = torch.randint(-3, 4, (64, 128), generator=g).half()
    x = torch.randint(-3, 4, (2, 9, 128), generator=g).half()
    bias = torch.randint(-3, 4, (64,), generator=g).half()
    mask = oracle.prune24_mask(w)
    wm = torch.where(mask, w, torch.zeros_like(w))
    s = sparse.to_sparse_semi_structured(w.to(cuda))
    ref = oracle.linear_ref(x, wm, bias)
    out = sparse.sparse_semi_structured_linear(x.to(cuda), s, bias=bias.to(cuda))
    assert out.float().cpu().equal(ref)
    out = sparse.sparse_semi_structured_linear(x.to(cuda), s.values(), s.indices(), bias=bias.to(cuda), activation="relu")
    assert out.float().cpu().equal(ref.clamp_min(0))
    out = sparse.sparse_semi_structured_linear(x.to(cuda), s, activation="silu")
    ref_silu = F.silu(oracle.linear_ref(x, wm))
    assert torch.allclose(out.float().cpu(), ref_silu, rtol=2e-3, atol=2e-3)
    out = sparse.sparse_semi_structured_linear(x.to(cuda), s, activation="gelu")          # exact (erf) GELU
    assert torch.allclose(out.float().cpu(), F.gelu(oracle.linear_ref(x, wm)), rtol=2e-3, atol=2e-3)
    with pytest.raises(RuntimeError):
        sparse.sparse_semi_structured_linear(x.to(cuda), s, activation="tanh")


def test_my_linear_and_sparse_linear_modules(cuda):
    """sparse/sparse_ops.py: MyLinear is nn.Linear; SparseLinear has the same forward and weight/bias
    gradients, and dX = dY . MVUE24(W^T)^T with the uniforms of torch's generator."""
    import sparse
    torch.manual_seed(3)
    ref = torch.nn.Linear(128, 64).to(cuda)
    x = torch.randn(8, 16, 128, device=cuda)
    gy = torch.randn(8, 16, 64, device=cuda)
    for cls in (sparse.MyLinear, sparse.SparseLinear):
        mod = cls(128, 64).to(cuda)
        mod.load_state_dict(ref.state_dict())
        xr, xm = x.clone().requires_grad_(), x.clone().requires_grad_()
        yr, ym = ref(xr), mod(xm)
        assert torch.allclose(ym, yr, atol=1e-5, rtol=1e-5)
        ref.zero_grad()
        yr.backward(gy)
        torch.manual_seed(11)
        ym.backward(gy)
        assert torch.allclose(mod.weight.grad, ref.weight.grad, atol=1e-4, rtol=1e-4)
        assert torch.allclose(mod.bias.grad, ref.bias.grad, atol=1e-4, rtol=1e-4)
        if cls is sparse.MyLinear:
            assert torch.allclose(xm.grad, xr.grad, atol=1e-5, rtol=1e-5)
        else:
            torch.manual_seed(11)
            w_est = sparse.MVUE24_approx_triton(mod.weight.detach().t()).t()
            want = (gy.reshape(-1, 64) @ w_est).view_as(x)
            assert torch.allclose(xm.grad, want, atol=1e-5, rtol=1e-5)
            assert ((w_est != 0).t().reshape(-1, 4).sum(-1) <= 2).all()        # 2:4 along the output axis


def test_soft_threshold_linear_module(cuda):
    """README S-STE recipe: forward uses scale * soft_threshold24(W); the gradient passes straight
    through to W; init_scale is the least-squares scale."""
    import sparse
    torch.manual_seed(4)
    mod = sparse.SoftThresholdLinear(128, 64).to(cuda)
    mod.init_scale()
    w = mod.weight.detach()
    ws, _ = oracle.soft_threshold24(w.cpu())
    want_scale = (w.cpu().flatten() @ ws.flatten()) / (ws.flatten() @ ws.flatten())
    assert abs(mod.scale.item() - want_scale.item()) < 1e-5 and mod.scale.item() > 1.0
    x = torch.randn(32, 128, device=cuda)
    y = mod(x)
    want = F.linear(x, ws.to(cuda) * mod.scale, mod.bias)
    assert torch.allclose(y, want, atol=1e-5, rtol=1e-5)
    gy = torch.randn_like(y)
    y.backward(gy)
    assert torch.allclose(mod.weight.grad, gy.t() @ x, atol=1e-4, rtol=1e-4)     # straight-through
    # STEP recipe: magnitude-pruned weight with a straight-through gradient
    w2 = torch.randn(64, 128, device=cuda, requires_grad=True)
    sp = sparse.Sparse24.apply(w2)
    want_sp, _ = oracle.sparse24_dense(w2.detach().cpu())
    assert sp.detach().cpu().equal(want_sp)
    sp.backward(torch.ones_like(sp))
    assert w2.grad.equal(torch.ones_like(w2))


@pytest.mark.parametrize("gdt", [torch.float32, torch.float16])
def test_masked_decay_adamw_kernel(cuda, gdt):
    """One fused pass against the oracle (float32; rtol 2e-6: torch's CPU ops may contract a
    multiply-add that the kernel rounds twice) and against the two-pass recipe it replaces."""
    import sparse
    g = torch.Generator().manual_seed(31)
    hyp = dict(lr=3e-3, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.1)
    p0 = torch.randn(96, 200, generator=g)                      # 19200 elements + odd tail coverage below
    mask = torch.rand(96, 200, generator=g) > 0.5
    par = torch.nn.Parameter(p0.clone().to(cuda))
    par.mask, par.mode, par.cnt = mask.to(cuda), "sparse", 3
    plain = torch.nn.Parameter(torch.randn(1003, generator=g).to(cuda))        # no mask, unaligned tail
    if gdt != torch.float32:
        par.grad_dtype = plain.grad_dtype = None                 # let the float32 parameters hold half gradients
    opt = sparse.MaskedDecayAdamW([par, plain], alpha=2e-4, **hyp)
    ref_par = torch.nn.Parameter(p0.clone().to(cuda))
    ref_plain = torch.nn.Parameter(plain.detach().clone())
    ref_opt = torch.optim.AdamW([ref_par, ref_plain], foreach=False, fused=False, **hyp)
    p, m, v = p0.clone(), torch.zeros_like(p0), torch.zeros_like(p0)
    q, qm, qv = plain.detach().cpu().clone(), torch.zeros(1003), torch.zeros(1003)
    for step in range(1, 5):
        grad = torch.randn(96, 200, generator=g).to(gdt)
        grad2 = torch.randn(1003, generator=g).to(gdt)
        par.grad, plain.grad = grad.to(cuda), grad2.to(cuda)
        opt.step()
        assert par.cnt == 0
        p, m, v = oracle.adamw_masked_decay(p, grad, m, v, mask, step, alpha=2e-4, **hyp)
        q, qm, qv = oracle.adamw_masked_decay(q, grad2, qm, qv, None, step, **hyp)
        assert torch.allclose(par.detach().cpu(), p, rtol=2e-6, atol=1e-8)
        assert torch.allclose(opt.state[par]["exp_avg"].cpu(), m, rtol=2e-6, atol=1e-10)
        assert torch.allclose(opt.state[par]["exp_avg_sq"].cpu(), v, rtol=2e-6, atol=1e-12)
        assert torch.allclose(plain.detach().cpu(), q, rtol=2e-6, atol=1e-8)
        # the recipe it replaces: masked_add_ on the float32 gradient, then an AdamW step
        ref_par.grad = grad.to(cuda).float()
        sparse.masked_add_(ref_par.grad, ref_par.data, par.mask, alpha=2e-4)
        ref_plain.grad = grad2.to(cuda).float()
        ref_opt.step()
        assert torch.allclose(par.detach(), ref_par.detach(), rtol=1e-5, atol=1e-7)
        assert torch.allclose(plain.detach(), ref_plain.detach(), rtol=1e-5, atol=1e-7)


@pytest.mark.parametrize("gdt,mdt,device_step", [(torch.float32, torch.bool, False), (torch.float16, torch.float32, True)])
def test_masked_decay_adamw_list_of_tensors(cuda, gdt, mdt, device_step):
    """A group of more tensors than one launch takes (56), with the lengths around a block of 1024 elements, a tensor
    whose storage starts off a 16-byte boundary, masked and unmasked ones mixed: two updates against the oracle
    (float32; rtol 2e-6 as above).  A tensor of another step count goes with the others of its own."""
    import sparse
    g = torch.Generator().manual_seed(32)
    hyp = dict(lr=3e-3, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.1)
    lengths = [1, 3, 4, 1020, 1023, 1024, 1025, 2048, 4096, 4099] * 6
    params, refs = [], []
    for i, n in enumerate(lengths):
        flat = torch.randn(n + 1, generator=g).to(cuda)
        p = torch.nn.Parameter(flat[1:] if i % 7 == 3 else flat[:-1])          # 4 bytes off a 16-byte boundary: single accesses
        p.grad_dtype = None
        mask = None
        if i % 3:
            mask = torch.rand(n, generator=g) > 0.5
            p.mask, p.mode = mask.to(cuda).to(mdt), "sparse"
        params.append(p)
        refs.append([p.detach().cpu().clone(), torch.zeros(n), torch.zeros(n), mask, 0])
    opt = sparse.MaskedDecayAdamW(params, alpha=2e-4, capturable=device_step, **hyp)
    for update in range(2):
        for i, (p, r) in enumerate(zip(params, refs)):
            if update == 0 and i == 5:
                p.grad = None                                                  # one update behind the others from here on
                continue
            grad = torch.randn(len(r[0]), generator=g).to(gdt)
            p.grad = grad.to(cuda)
            r[4] += 1
            r[0], r[1], r[2] = oracle.adamw_masked_decay(r[0], grad, r[1], r[2], r[3], r[4], alpha=2e-4, **hyp)
        opt.step()
    for p, (want, m, v, _, step) in zip(params, refs):
        assert torch.allclose(p.detach().cpu(), want, rtol=2e-6, atol=1e-8)
        assert torch.allclose(opt.state[p]["exp_avg"].cpu(), m, rtol=2e-6, atol=1e-10)
        assert torch.allclose(opt.state[p]["exp_avg_sq"].cpu(), v, rtol=2e-6, atol=1e-12)
        assert int(opt.state[p]["step"]) == step


def test_masked_decay_adamw_moments_after_a_refused_gradient(cuda):
    """A first step that is refused because of a later tensor leaves nothing behind: the moments start from zero afterwards."""
    import sparse
    first = [torch.nn.Parameter(torch.ones(64, 32, device=cuda)) for _ in range(2)]
    opt = sparse.MaskedDecayAdamW(first, lr=1e-2)
    first[0].grad = torch.full_like(first[0], 0.5)
    first[1].grad = torch.full((32, 64), 0.5, device=cuda).t()
    junk = [torch.full((64, 32), float("nan"), device=cuda) for _ in range(8)]       # what fresh memory may hold
    del junk
    with pytest.raises(RuntimeError, match="strides"):
        opt.step()
    first[1].grad = first[0].grad.clone()
    opt.step()
    want, m, v = oracle.adamw_masked_decay(torch.ones(64, 32), torch.full((64, 32), 0.5), torch.zeros(64, 32), torch.zeros(64, 32), None, 1, alpha=0.0,
                                           lr=1e-2, betas=opt.defaults["betas"], eps=opt.defaults["eps"], weight_decay=opt.defaults["weight_decay"])
    for p in first:                                                                  # float32 arithmetic of a few operations
        assert torch.allclose(p.detach().cpu(), want, rtol=2e-6, atol=1e-8)
        assert torch.allclose(opt.state[p]["exp_avg"].cpu(), m, rtol=2e-6, atol=1e-10)


@pytest.mark.parametrize("capturable", [False, True])
def test_masked_decay_adamw_shared_storage(cuda, capturable):
    """Two parameters on the same memory are updated one after the other, as by one launch each."""
    import sparse
    torch.manual_seed(3)
    base = torch.randn(300, 512, device=cuda)
    results = []
    for grouped in (True, False):
        data = base.clone()
        params = [torch.nn.Parameter(data), torch.nn.Parameter(torch.ones(7, device=cuda)), torch.nn.Parameter(data)]
        for i, p in enumerate(params):
            p.grad = torch.full_like(p, 0.25 * (i + 1))
        groups = [params] if grouped else [[p] for p in params]
        opts = [sparse.MaskedDecayAdamW(g, lr=1e-2, weight_decay=0.1, capturable=capturable) for g in groups]
        for _ in range(2):
            for opt in opts:
                opt.step()
        results.append([p.detach().clone() for p in params])
    for a, b in zip(*results):
        assert a.equal(b)


@pytest.mark.parametrize("capturable", [False, True])
@pytest.mark.parametrize("starts", [(0, 4), (513, 0), (0, 1024)])
def test_masked_decay_adamw_overlapping_parameters(cuda, capturable, starts):
    """Parameters that are overlapping parts of one buffer are updated one after the other, as by one optimizer each."""
    import sparse
    torch.manual_seed(4)
    base = torch.randn(150000, device=cuda)
    results = []
    for grouped in (True, False):
        data = base.clone()
        params = [torch.nn.Parameter(data[start:]) for start in starts + starts[:1]]
        for i, p in enumerate(params):
            p.grad = torch.full_like(p, 0.25 * (i + 1))
        groups = [params] if grouped else [[p] for p in params]
        opts = [sparse.MaskedDecayAdamW(g, lr=1e-2, weight_decay=0.1, capturable=capturable) for g in groups]
        for _ in range(2):
            for opt in opts:
                opt.step()
        results.append(data)
    assert results[0].equal(results[1])


@pytest.mark.parametrize("gdt", [torch.float32, torch.bfloat16])
def test_masked_decay_adamw_step_count_on_the_device(cuda, gdt):
    """capturable=True: the step count is an int64 in device memory and the bias corrections 1 - beta^step are
    formed by the kernel.  Twelve updates must leave parameters and moments bit-equal to the optimizer with the
    count on the host (same double-precision formulas, rounded to float32 at the same places), for a masked
    parameter and an unmasked one with an odd length; then a single update recorded into a HIP graph and replayed
    three times must continue the same sequence (a recording with the count frozen in it would not)."""
    import sparse
    g = torch.Generator().manual_seed(33)
    hyp = dict(lr=3e-3, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.1, alpha=2e-4)
    p0, q0 = torch.randn(96, 200, generator=g), torch.randn(1003, generator=g)
    mask = (torch.rand(96, 200, generator=g) > 0.5).to(cuda)
    models = []
    for capturable in (False, True):
        par, plain = torch.nn.Parameter(p0.clone().to(cuda)), torch.nn.Parameter(q0.clone().to(cuda))
        par.mask, par.mode, par.cnt = mask, "sparse", 0
        if gdt != torch.float32:
            par.grad_dtype = plain.grad_dtype = None
        par.grad, plain.grad = torch.zeros(96, 200, device=cuda, dtype=gdt), torch.zeros(1003, device=cuda, dtype=gdt)
        models.append((par, plain, sparse.MaskedDecayAdamW([par, plain], capturable=capturable, **hyp)))
    (hp, hq, hopt), (dp, dq, dopt) = models

    def same(step):
        for a, b in ((hp, dp), (hq, dq)):
            assert torch.equal(a, b), step
            assert torch.equal(hopt.state[a]["exp_avg"], dopt.state[b]["exp_avg"]), step
            assert torch.equal(hopt.state[a]["exp_avg_sq"], dopt.state[b]["exp_avg_sq"]), step
            assert int(dopt.state[b]["step"]) == hopt.state[a]["step"] == step

    grads = [(torch.randn(96, 200, generator=g).to(gdt).to(cuda), torch.randn(1003, generator=g).to(gdt).to(cuda)) for _ in range(15)]
    for step in range(1, 13):
        for par, plain, opt in models:
            par.grad.copy_(grads[step - 1][0]); plain.grad.copy_(grads[step - 1][1])
            opt.step()
        same(step)
    assert dopt.state[dp]["step"].is_cuda and dopt.state[dp]["step"].dtype == torch.int64
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        dopt.step()
    for step in range(13, 16):
        dp.grad.copy_(grads[step - 1][0]); dq.grad.copy_(grads[step - 1][1])
        graph.replay()
        hp.grad.copy_(grads[step - 1][0]); hq.grad.copy_(grads[step - 1][1])
        hopt.step()
        torch.cuda.synchronize()
        same(step)


@pytest.mark.parametrize("capturable", [False, True])
def test_masked_decay_adamw_resumes_from_a_state_dict(cuda, capturable):
    """Three updates, the state through a checkpoint on the host, two more: the bits of five updates in a row."""
    import io
    import sparse
    grads = torch.randn(5, 1003, generator=torch.Generator().manual_seed(5)).to(cuda)

    def updates(p, opt, which):
        for i in which:
            p.grad = grads[i].clone()
            opt.step()

    def fresh(data):
        p = torch.nn.Parameter(data.clone())
        return p, sparse.MaskedDecayAdamW([p], lr=1e-2, weight_decay=0.1, capturable=capturable)

    start = torch.ones(1003, device=cuda)
    whole, opt = fresh(start)
    updates(whole, opt, range(5))
    first, opt_first = fresh(start)
    updates(first, opt_first, range(3))
    blob = io.BytesIO()
    torch.save(opt_first.state_dict(), blob)
    blob.seek(0)
    second, opt_second = fresh(first.detach())
    opt_second.load_state_dict(torch.load(blob, map_location="cpu", weights_only=True))
    updates(second, opt_second, range(3, 5))
    assert second.equal(whole)
    assert int(opt_second.state[second]["step"]) == 5 and opt_second.state[second]["exp_avg_sq"].equal(opt.state[whole]["exp_avg_sq"])


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-6), (torch.float16, 1e-3), (torch.bfloat16, 8e-3)])
@pytest.mark.parametrize("shape", [(4, 32, 256), (3, 5, 24), (2, 7, 10), (1, 1, 2)])
@pytest.mark.parametrize("transposed", [False, True])
def test_gelu_glu_forward_backward(cuda, dtype, tol, shape, transposed):
    """GELUglu against the float64 oracle.  Tolerances: float32 arithmetic then one rounding to the
    storage type, so 2e-6 (float32), 2^-10 (float16) and 2^-7 (bfloat16) of the largest
    magnitude; `transposed` stores the last dimension strided (the reference's 2-d path)."""
    import sparse
    g = torch.Generator().manual_seed(41)
    a, b, c = shape
    inp = (2 * torch.randn(a * b, c, generator=g)).to(dtype)
    go = torch.randn(a * b, c // 2, generator=g).to(dtype)
    dev_in = inp.to(cuda)
    if transposed:
        dev_in = dev_in.t().contiguous().t()                    # same values, column-major storage
    dev_in = dev_in.view(a, b, c).requires_grad_(True)
    out = sparse.GELUglu()(dev_in)
    want = oracle.gelu_glu_forward(inp.view(a, b, c))
    assert out.shape == (a, b, c // 2) and out.dtype == dtype
    scale = want.abs().max().item()
    assert (out.double().cpu() - want).abs().max().item() <= tol * scale + 1e-30
    out.backward(go.to(cuda).view(a, b, c // 2))
    want_g = oracle.gelu_glu_backward(go.view(a, b, c // 2), inp.view(a, b, c))
    assert dev_in.grad.shape == (a, b, c) and dev_in.grad.dtype == dtype
    gscale = want_g.abs().max().item()
    assert (dev_in.grad.double().cpu() - want_g).abs().max().item() <= tol * gscale + 1e-30


def test_gelu_glu_errors(cuda):
    import sparse
    with pytest.raises(RuntimeError):
        sparse.gelu_glu.apply(torch.zeros(2, 3, 5, device=cuda))          # odd last dimension
    with pytest.raises(RuntimeError):
        sparse.gelu_glu.apply(torch.zeros(2, 3, 4))                       # not on the GPU
    with pytest.raises(AssertionError):
        sparse.gelu_glu.apply(torch.zeros(6, 4, device=cuda))             # the reference asserts a 3-d input


@pytest.mark.parametrize("grad_dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("amsgrad", [False, True])
@pytest.mark.parametrize("n,offset", [(4096, 0), (1031, 0), (2050, 1)])
def test_adamw_step_kernel_matches_oracle(cuda, grad_dtype, amsgrad, n, offset):
    """tf24_adamw_step against the oracle over several steps, both phases, with the variance-change
    partial sums; `offset` shifts the tensors off 16-byte alignment (scalar-access variant).
    Tolerance 2e-6 relative: float32 arithmetic, torch may contract the oracle's multiply-adds."""
    from sparse import _native as N
    lib = N.lib()
    g = torch.Generator().manual_seed(61)
    hp = dict(lr=2e-3, betas=(0.9, 0.98), eps=1e-7, weight_decay=0.02)

    def dev(t):                                   # a view that starts `offset` elements into its buffer
        buf = torch.zeros(t.numel() + 8, dtype=t.dtype, device=cuda)
        buf[offset:offset + t.numel()] = t.to(cuda)
        return buf[offset:offset + t.numel()]

    p = torch.randn(n, generator=g)
    m, v = torch.zeros(n), torch.zeros(n)
    vmax = torch.zeros(n) if amsgrad else None
    dp, dm, dv = dev(p), dev(m), dev(v)
    dx = dev(vmax) if amsgrad else None
    nz = lib.tf24_adamw_step_partials(n)
    assert nz == (n + 1023) // 1024
    frozen = None
    for step in range(1, 6):
        grad = (torch.randn(n, generator=g) * (1.5 if step % 2 else 0.3)).to(grad_dtype)
        dg = dev(grad)
        phase2 = step >= 4
        if phase2 and frozen is None:
            frozen = (vmax if amsgrad else v).clone()
            dfrozen = dev(frozen)
        for option in ([2, 1] if step == 2 else [1]):       # option 2 runs on copies first: the update itself is the same
            z = torch.full((nz,), float("nan"), dtype=torch.float32, device=cuda)
            args = [t.clone() for t in (dp, dm, dv)] if option == 2 else [dp, dm, dv]
            N.check(lib.tf24_adamw_step(
                args[0].data_ptr(), dg.data_ptr(), N.dtype_code(grad_dtype), args[1].data_ptr(), args[2].data_ptr(),
                (dx.clone() if option == 2 else dx).data_ptr() if amsgrad else None, dfrozen.data_ptr() if phase2 else None,
                n, hp["lr"], hp["betas"][0], hp["betas"][1], hp["eps"], hp["weight_decay"], step,
                None if phase2 else z.data_ptr(), 0 if phase2 else option, N.stream_ptr()))
            if not phase2:
                _, _, _, _, change = oracle.adamw_step_update(p, grad, m, v, step, max_exp_avg_sq=vmax, **hp)
                want_z = oracle.variance_change_statistic([change], option=option)
                got = z.double().sum().item() / n
                got = got if option == 1 else torch.exp(torch.tensor(got, dtype=torch.float64)).item()
                assert abs(got - want_z) <= 2e-5 * abs(want_z) + 1e-12, (step, option, got, want_z)
        p, m, v, vmax, _ = oracle.adamw_step_update(p, grad, m, v, step, max_exp_avg_sq=vmax,
                                                    precond_variance=frozen if phase2 else None, **hp)
        for got, want in ((dp, p), (dm, m), (dv, v)) + (((dx, vmax),) if amsgrad else ()):
            assert torch.allclose(got.cpu(), want, rtol=2e-6, atol=1e-9), step


def test_adamw_step_optimizer_phases(cuda):
    """The AdamW_STEP class: watches only parameters carrying `mask`, switches at t > T_max, freezes the
    variance, and from then on divides tracked parameters by it; untracked ones stay on AdamW."""
    import sparse
    torch.manual_seed(62)
    w = torch.nn.Parameter(torch.randn(48, 40, device=cuda))
    b = torch.nn.Parameter(torch.randn(40, device=cuda))
    w.mask = 'dense'
    hp = dict(lr=1e-2, betas=(0.9, 0.5), eps=1e-8, weight_decay=0.01)
    opt = sparse.AdamW_STEP([w, b], clipping=(1, 3), option=1, **hp)
    assert opt.T_omega == 2 and opt.mask == 'dense'
    ow, ob = w.detach().cpu().clone(), b.detach().cpu().clone()
    mw, vw, mb, vb = torch.zeros_like(ow), torch.zeros_like(ow), torch.zeros_like(ob), torch.zeros_like(ob)
    frozen = None
    g = torch.Generator().manual_seed(63)
    for t in range(1, 7):
        gw, gb = torch.randn(48, 40, generator=g), torch.randn(40, generator=g)
        w.grad, b.grad = gw.to(cuda), gb.to(cuda)
        opt.step()
        ow, mw, vw, _, change = oracle.adamw_step_update(ow, gw, mw, vw, t, precond_variance=frozen, **hp)
        ob, mb, vb, _, _ = oracle.adamw_step_update(ob, gb, mb, vb, t, **hp)
        assert torch.allclose(w.detach().cpu(), ow, rtol=3e-6, atol=1e-8), t
        assert torch.allclose(b.detach().cpu(), ob, rtol=3e-6, atol=1e-8), t
        if t <= 3:
            assert opt.mask == 'dense' and w.mask == 'dense' and len(opt.sliding_window) == min(t, 2)
            z = oracle.variance_change_statistic([change], option=1)
            assert abs(opt.sliding_window[-1].item() - z) <= 1e-5 * z
        elif t == 4:                                                      # t > T_max = 3: switched after this update
            assert opt.mask == 'sparse' and w.mask == 'sparse'
            frozen = vw.clone()
            assert torch.allclose(opt.state[w]['preconditioned_variance'].cpu(), frozen, rtol=3e-6, atol=1e-12)
            assert 'preconditioned_variance' not in opt.state[b]
    assert opt.t == 6 and len(opt.sliding_window) == 2                    # the window stops growing after the switch
    with pytest.raises(ValueError):
        sparse.AdamW_STEP([w], option=3)


def test_entry_points_under_graph_capture(cuda):
    """The library only launches kernels on the stream it is given (no allocation, no synchronisation,
    no memset), so its calls can be recorded into a HIP graph: compression, both matmul forms (the
    split one with its workspace and reduction) and the masked decay are captured once and replayed
    on new contents of the same buffers, with eager work between the replays; every replay must give
    the bits of the eager calls."""
    import sparse
    n, k, m = 512, 4096, 48
    gen = torch.Generator().manual_seed(71)
    w = torch.randn(n, k, generator=gen).half().to(cuda)
    x = torch.randn(m, k, generator=gen).half().to(cuda)
    g32 = torch.randn(n, k, generator=gen).to(cuda)

    def work():
        s = sparse.to_sparse_semi_structured(w)                     # magnitude rule: no random numbers
        y = torch.mm(x, s.t())                                      # few dense columns: k pieces + reduction
        z = torch.mm(s, w.t())                                      # [n, n]: k-strided dense operand
        grad = g32.clone()
        sparse.masked_add_(grad, w.float(), (s.to_dense() != 0), alpha=2e-4)
        return y, z, grad

    work()                                                          # warm up outside the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            captured = work()
    torch.cuda.synchronize()
    for it in range(3):
        w.copy_(torch.randn(n, k, generator=gen).half())
        x.copy_(torch.randn(m, k, generator=gen).half())
        g32.copy_(torch.randn(n, k, generator=gen))
        eager = [t.clone() for t in work()]
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for name, a, b in zip(("x @ S.t", "S @ w.t", "masked decay"), captured, eager):
            assert torch.equal(a, b), (it, name)


@pytest.mark.parametrize("tokens,m,n", [(1, 8, 8), (31, 264, 40), (32, 256, 256), (33, 512, 264), (65, 248, 1000), (96, 256, 8),
                                        (128, 8, 256), (129, 768, 512), (161, 256, 256), (1000, 3072, 768), (4099, 768, 3072),
                                        (33, 192, 192), (65, 200, 384), (65, 4104, 3080), (2308, 240, 456), (3189, 256, 208)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_grad_weight_kernel(cuda, tokens, m, n, dtype):
    """dY^T x and sum(dY) of the dense layers' kernel, with as many pieces of the token axis as it likes, in one piece, with and
    without the sums, and from rows with a pitch; columns and tokens that fill no tile or stage; the last three are products for 256 x 256 tiles, the others for 192 x 192 ones.
    Bound: a float32 sum of `tokens` exact products in any order errs by at most tokens * 2^-23 times the sum of their
    magnitudes, and is rounded once to 11 (8) bits."""
    from sparse import _native as N
    gen = torch.Generator(device=cuda).manual_seed(tokens * 7 + m + n)
    g = torch.randn(tokens, m + 16, device=cuda, generator=gen).to(dtype)[:, 8:8 + m]
    x = torch.randn(tokens, n, device=cuda, generator=gen).to(dtype)
    lib = N.lib()
    nbytes = lib.tf24_grad_weight_workspace_bytes(tokens, m, n)
    gt, xd = g.double().t().contiguous(), x.double()
    half_ulp = 2.0 ** (-11 if dtype == torch.float16 else -8)
    for want, size, name in ((gt @ xd, gt.abs() @ xd.abs(), "dW"), (gt.sum(1), gt.abs().sum(1), "db")):
        limit = want.abs() * half_ulp + size * tokens * 2.0 ** -23 + 1e-7
        for bytes_given in {0, nbytes}:
            for with_bias in (True, False):
                ws = torch.empty(max(bytes_given, 16), dtype=torch.uint8, device=cuda)
                dw = torch.full((m, n), float("nan"), dtype=dtype, device=cuda)
                db = torch.full((m,), float("nan"), dtype=dtype, device=cuda)
                N.check(lib.tf24_grad_weight(g.data_ptr(), g.stride(0), x.data_ptr(), x.stride(0), N.dtype_code(dtype), tokens, m, n, dw.data_ptr(),
                                             db.data_ptr() if with_bias else None, ws.data_ptr(), bytes_given, N.stream_ptr()))
                if name == "db" and not with_bias:
                    assert db.isnan().all()
                else:
                    got = dw if name == "dW" else db
                    assert ((got.double() - want).abs() <= limit).all(), (name, bytes_given, with_bias)


@pytest.mark.parametrize("tokens,m,n", [(1, 8, 8), (31, 264, 40), (65, 248, 1000), (129, 768, 512), (1000, 3072, 768), (4099, 768, 3072), (12287, 520, 264)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_grad_weight_kernel_is_exact_and_deterministic(cuda, tokens, m, n, dtype):
    """Small integers, whose sums float32 holds exactly in any order: dW and db are those sums rounded once, whatever the number
    of pieces (partial sums of 16 bits would not be).  Random operands: the same bits again, and an error of about
    sqrt(tokens) roundings of sums of that size (8 standard deviations of them) beside the one to 16 bits."""
    from sparse import _native as N
    gen = torch.Generator(device=cuda).manual_seed(tokens + m + n)
    lib = N.lib()
    nbytes = lib.tf24_grad_weight_workspace_bytes(tokens, m, n)
    ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=cuda)

    def run(g, x, bytes_given):
        dw, db = torch.empty((m, n), dtype=dtype, device=cuda), torch.empty((m,), dtype=dtype, device=cuda)
        N.check(lib.tf24_grad_weight(g.data_ptr(), m, x.data_ptr(), n, N.dtype_code(dtype), tokens, m, n, dw.data_ptr(), db.data_ptr(),
                                     ws.data_ptr(), bytes_given, N.stream_ptr()))
        return dw, db

    g, x = (torch.randint(-8, 9, (tokens, c), device=cuda, generator=gen).to(dtype) for c in (m, n))
    want = (g.double().t().contiguous() @ x.double()).to(dtype), g.double().sum(0).to(dtype)
    for bytes_given in {0, nbytes}:
        for got, exact in zip(run(g, x, bytes_given), want):
            assert got.equal(exact), bytes_given
    g, x = (torch.randn(tokens, c, device=cuda, generator=gen).to(dtype) for c in (m, n))
    exact = g.double().t().contiguous() @ x.double(), g.double().sum(0)
    half_ulp = 2.0 ** (-11 if dtype == torch.float16 else -8)
    for bytes_given in {0, nbytes}:
        first = run(g, x, bytes_given)
        wide = torch.empty((m, n), device=cuda), torch.empty((m,), device=cuda)          # the float32 form: the same values
        N.check(lib.tf24_grad_weight_f32(g.data_ptr(), m, x.data_ptr(), n, N.dtype_code(dtype), tokens, m, n, wide[0].data_ptr(), wide[1].data_ptr(),
                                         ws.data_ptr(), bytes_given, N.stream_ptr()))
        assert all(a.equal(b.float()) for a, b in zip(wide, first))
        for got, again, ref in zip(first, run(g, x, bytes_given), exact):
            assert got.equal(again), bytes_given
            # each of the `tokens` additions rounds a partial sum of at most about 4 sqrt(tokens) by half of 2^-23 of it
            limit = ref.abs() * half_ulp + 8 * tokens ** 0.5 * (4 * tokens ** 0.5) * 2.0 ** -24 + 2.0 ** -25
            assert bool(((got.double() - ref).abs() <= limit).all()), bytes_given


@pytest.mark.parametrize("tokens,bias,dtype", [((300,), True, torch.bfloat16), ((5, 41), True, torch.float16), ((4100,), False, torch.bfloat16),
                                               ((3, 200), False, torch.float16)])
def test_soft_threshold_linear_under_autocast(cuda, tokens, bias, dtype):
    """In mixed precision the module takes its own weight gradient (from a number of tokens on); the same as F.linear under
    autocast, also where a graph of the gradients, a tangent of the input or a mode asks for torch's operators."""
    import sparse
    torch.manual_seed(8)
    mod = sparse.SoftThresholdLinear(128, 264, bias=bias, device=cuda)
    mod.init_scale()
    params = list(mod.parameters())
    x = torch.randn(*tokens, 128, device=cuda, requires_grad=True)
    gy = torch.randn(*tokens, 264, device=cuda).to(dtype)

    def grads(y, **kw):
        return [y] + list(torch.autograd.grad(y, [x] + params, gy, **kw))

    with torch.autocast("cuda", dtype=dtype):
        y_ref = F.linear(x, mod.get_sparse_weights(), mod.bias)
        y = mod(x)
    assert "linear16" in type(y.grad_fn).__name__
    want = grads(y_ref)
    # one rounding to 16 bits each, of sums that differ in order: at most a unit in the last place where they straddle a boundary
    tol = 2.0 ** (-10 if dtype == torch.float16 else -7)
    for a, b in zip(grads(y, retain_graph=True), want):
        assert a.dtype == b.dtype and torch.allclose(a.float(), b.float(), rtol=tol, atol=1e-4)
    if dtype == torch.float16:                                                      # gradients that autograd maps over
        mapped = torch.autograd.grad(y, params, torch.stack([gy, -2 * gy]), is_grads_batched=True, retain_graph=True)
        for got, b in zip(mapped, want[2:]):
            assert torch.allclose(got[0].float(), b.float(), rtol=tol, atol=1e-4) and torch.allclose(got[1].float(), -2 * b.float(), rtol=tol, atol=2e-4)
    first = grads(y, create_graph=True)
    assert first[1].grad_fn is not None
    torch.autograd.grad(first[1].float().sum(), params[0])                          # reaches the weight through dX
    with torch.autograd.forward_ad.dual_level(), torch.autocast("cuda", dtype=dtype):
        dual = torch.autograd.forward_ad.make_dual(x.detach(), torch.ones_like(x))
        tangent = torch.autograd.forward_ad.unpack_dual(mod(dual)).tangent
    assert tangent is not None


@pytest.mark.parametrize("tokens,bias", [(40, True), (300, True), (300, False), (4100, False)])
def test_soft_threshold_linear_backward_inside_autocast(cuda, tokens, bias):
    """The backward pass gives the same bits outside autocast, inside it, and inside it with another type."""
    import sparse
    torch.manual_seed(9)
    mod = sparse.SoftThresholdLinear(128, 264, bias=bias, device=cuda)
    mod.init_scale()
    x = torch.randn(tokens, 128, device=cuda, requires_grad=True)
    gy = torch.randn(tokens, 264, device=cuda).bfloat16()
    wanted = [x] + list(mod.parameters())
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = mod(x)
        inside = torch.autograd.grad(y, wanted, gy, retain_graph=True)
    with torch.autocast("cuda", dtype=torch.float16):
        other = torch.autograd.grad(y, wanted, gy, retain_graph=True)
    for a, b, c in zip(torch.autograd.grad(y, wanted, gy), inside, other):
        assert a.dtype == torch.float32 and a.equal(b) and a.equal(c)


@pytest.mark.parametrize("tokens,bias", [(300, True), (4100, False)])
def test_soft_threshold_linear_backward_under_tangents_and_modes(cuda, tokens, bias):
    """A tangent of the output's gradient reaches the weight's and the bias's, and a dispatch mode around the backward pass sees
    the products, also where the forward pass ran without either."""
    import sparse
    from torch.autograd import forward_ad
    from torch.utils._python_dispatch import TorchDispatchMode
    torch.manual_seed(9)
    mod = sparse.SoftThresholdLinear(128, 264, bias=bias, device=cuda)
    mod.init_scale()
    params = list(mod.parameters())
    x = torch.randn(tokens, 128, device=cuda)
    gy, tangent = (torch.randn(tokens, 264, device=cuda).bfloat16() for _ in range(2))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = mod(x)
    assert "linear16" in type(y.grad_fn).__name__
    want, want_tangent = ([gy_.float().t() @ x.bfloat16().float()] + ([gy_.float().sum(0)] if bias else []) for gy_ in (gy, tangent))
    with forward_ad.dual_level():
        got = [forward_ad.unpack_dual(t) for t in torch.autograd.grad(y, params, forward_ad.make_dual(gy, tangent), retain_graph=True)]
        for t, a, b in zip(got, want, want_tangent):                      # one rounding to bfloat16 each, of sums in another order
            assert torch.allclose(t.primal, a, rtol=2 ** -7, atol=1e-2)
            assert t.tangent is not None and torch.allclose(t.tangent, b, rtol=2 ** -7, atol=1e-2)

    class Seen(TorchDispatchMode):
        names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(func.__name__)
            return func(*args, **(kwargs or {}))

    with Seen() as seen:
        torch.autograd.grad(y, params, gy)
    assert seen.names.count("mm.default") == 1                            # dW (x needs no gradient)


@pytest.mark.parametrize("n,m", [(8, (1 << 20) + 8), ((1 << 20) + 8, 8), (8, 1 << 20)])
def test_soft_threshold_linear_very_wide(cuda, n, m):
    """More features on either side than the weight-gradient kernel takes, and as many: the gradients of F.linear.  Exact:
    small integers, sums below 2^8 in magnitude."""
    import sparse
    mod = sparse.SoftThresholdLinear(n, m, device=cuda)
    mod.init_scale()
    g = torch.Generator(device=cuda).manual_seed(m)
    x = torch.randint(-1, 2, (256, n), device=cuda, generator=g).float()
    gy = (torch.randint(-1, 2, (256, m), device=cuda, generator=g) * (torch.rand(256, m, device=cuda, generator=g) < 0.3)).bfloat16()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = mod(x)
    grads = torch.autograd.grad(y, [mod.weight, mod.bias], gy)
    assert grads[0].equal(gy.float().t() @ x) and grads[1].equal(gy.float().sum(0))


def test_soft_threshold_linear_negated_bias(cuda):
    """A bias whose sign is still to be applied is not read as it lies.  Bit for bit the result of the bias with its sign."""
    import sparse
    torch.manual_seed(3)
    mod = sparse.SoftThresholdLinear(128, 264, device=cuda)
    mod.init_scale()
    x, bias = torch.randn(300, 128, device=cuda), torch.randn(264, device=cuda)
    call = lambda b: torch.func.functional_call(mod, {"bias": b}, (x,))
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        assert call(torch._neg_view(bias)).equal(call(-bias))


@pytest.mark.parametrize("shape", [(1, 8), (64, 128), (37, 1000), (768, 3072)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_soft_threshold16_is_threshold_scale_and_cast(cuda, shape, dtype):
    """Bit for bit, special values (and a negative scale, which makes dropped zeros negative) included."""
    import sparse
    from sparse.sparse_ops import _soft_threshold16
    torch.manual_seed(1)
    w = torch.randn(*shape, device=cuda) * torch.logspace(-9, 6, shape[1], device=cuda)
    w.view(-1)[:8] = torch.tensor([0.0, -0.0, float("inf"), 1.0, 2.0, 2.0, -2.0, 1e-42], device=cuda)
    for value, where in ((1.37, cuda), (-0.6, cuda), (-0.6, "cpu"), (1.37, "cpu")):      # (a layer made on the GPU keeps its scale on the host)
        scale = torch.tensor(value, device=where)
        want = (sparse.soft_threshold24(w)[0] * scale).to(dtype)
        got = _soft_threshold16.apply(w, scale, dtype)
        assert got.view(torch.int16).equal(want.view(torch.int16)) or (
            got.isnan().equal(want.isnan()) and got[~got.isnan()].view(torch.int16).equal(want[~want.isnan()].view(torch.int16)))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_sparse_linear_transpose_bias_may_change_before_the_backward_pass(cuda, dtype):
    """No gradient depends on the bias: one that has been updated in place since the forward pass, in either type, is no error."""
    import sparse
    torch.manual_seed(0)
    mod = sparse.SparseLinearTranspose(128, 64, device=cuda)
    bias = torch.nn.Parameter(torch.randn(64, device=cuda, dtype=dtype))
    mod.bias = bias
    x, gy = torch.randn(64, 128, device=cuda, dtype=torch.float16), torch.randn(64, 64, device=cuda, dtype=torch.float16)
    y = mod(x)
    with torch.no_grad():
        bias += 1
    y.backward(gy)
    assert bias.grad.dtype == dtype and torch.allclose(bias.grad.float(), gy.float().sum(0), rtol=1e-3, atol=1e-2)


@pytest.mark.parametrize("leaf", [True, False])
def test_soft_threshold_linear_lets_go_of_its_weight(cuda, leaf):
    """The layer's graph does not keep a float32 weight that is the result of something, and leads to it, or to a parameter, all
    the same: d(sum of dX) / dW is the straight-through sum of dY over the tokens, also where the weight changes in between."""
    import gc
    import weakref
    import sparse
    torch.manual_seed(11)
    mod = sparse.SoftThresholdLinear(128, 264, device=cuda)
    mod.init_scale()
    base = mod.weight
    x, gy = torch.randn(300, 128, device=cuda, requires_grad=True), torch.randn(300, 264, device=cuda).bfloat16()

    def forward():
        weight = base if leaf else base * 1.0
        with torch.autocast("cuda", dtype=torch.bfloat16):
            return torch.func.functional_call(mod, {"weight": weight}, (x,)), None if leaf else weakref.ref(weight)

    y, freed = forward()
    gc.collect()
    assert leaf or freed() is None
    with torch.no_grad():
        base.add_(1.0)
    dx, = torch.autograd.grad(y, x, gy, create_graph=True)
    second, = torch.autograd.grad(dx.float().sum(), base)
    want = gy.float().sum(0)[:, None].expand(264, 128)
    # (dX and its gradient are 16-bit products: 2^-8 of each sum of 300 terms of about 1)
    assert second.dtype == torch.float32 and torch.allclose(second, want, rtol=2.0 ** -7, atol=0.1)
    y, _ = forward()
    first = torch.autograd.grad(y, (x, base, mod.bias), gy, retain_graph=True)
    with torch.autograd.graph.save_on_cpu():
        y, _ = forward()
    assert all(a.equal(b) for a, b in zip(first, torch.autograd.grad(y, (x, base, mod.bias), gy)))


@pytest.mark.parametrize("rows,k,tokens", [(8, 256, 1), (192, 256, 192), (200, 320, 193), (184, 1536, 191), (768, 3072, 400), (2056, 512, 4100), (520, 6400, 777)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("strided", [False, True])
def test_dense_linear_kernel(cuda, rows, k, tokens, dtype, strided):
    """The S-STE layer's product with its weight and with its transpose: rows and tokens that fill no tile, the fewest stages, stages
    in another order per XCD (24 and more), tiles behind each other in one workgroup (2056 x 4100), operands and results with a pitch.
    Small integers, whose sums float32 holds exactly: rounded once.  Random operands: a float32 sum of k exact products and the bias in any
    order errs by at most (k + 1) * 2^-23 times the sum of their magnitudes, and is rounded once to 11 (8) bits."""
    from sparse import _native as N
    gen = torch.Generator(device=cuda).manual_seed(rows + k + tokens)
    shape = (k, rows + 8) if strided else (rows, k + 8)

    def run(w, x, bias):
        y = torch.full((tokens, rows + 8), float("nan"), dtype=dtype, device=cuda)
        N.check(N.lib().tf24_linear16(w.data_ptr(), w.stride(0), strided, x.data_ptr(), x.stride(0), N.dtype_code(dtype), rows, k, tokens, y.data_ptr(),
                                      y.stride(0), N.ptr(bias), N.stream_ptr()))
        assert y[:, rows:].isnan().all()
        return y[:, :rows]

    for ints in (True, False):
        draw = (lambda *s: torch.randint(-4, 5, s, device=cuda, generator=gen).to(dtype)) if ints else (lambda *s: torch.randn(*s, device=cuda, generator=gen).to(dtype))
        w, x, bias = draw(*shape), draw(tokens, k + 16)[:, 8:8 + k], draw(rows)
        wk = (w[:, :rows].t() if strided else w[:, :k]).double().contiguous()
        for b in (None, bias):
            want = x.double() @ wk.t().contiguous() + (0 if b is None else b.double())
            got = run(w, x, b)
            if ints:
                assert got.equal(want.to(dtype))
            else:
                size = x.double().abs() @ wk.abs().t().contiguous() + (0 if b is None else b.double().abs())
                limit = want.abs() * 2.0 ** (-11 if dtype == torch.float16 else -8) + size * (k + 1) * 2.0 ** -23 + 1e-7
                assert ((got.double() - want).abs() <= limit).all()
                assert got.equal(run(w, x, b))


@pytest.mark.parametrize("rows,k,tokens", [(3072, 768, 800), (768, 3072, 800), (2048, 512, 1500)])
def test_soft_threshold_layer_products_take_the_kernel(cuda, rows, k, tokens, monkeypatch):
    """One round of tiles or part of one: an S-STE layer's product and input gradient are the same where the kernel takes them as in the
    library (two float32 sums of n terms, rounded to 8 bits), infinite activations included; gradients with another order take it too."""
    from sparse import _native as N, SoftThresholdLinear
    import torch.nn.functional as F
    gen = torch.Generator(device=cuda).manual_seed(rows)
    layer = SoftThresholdLinear(k, rows, device=cuda)
    layer.init_scale()
    x = torch.randn(2, tokens // 2, k, device=cuda, generator=gen).requires_grad_()
    dy = torch.randn(2, tokens // 2, rows, device=cuda, generator=gen).bfloat16()
    x.data[1, 3, 5] = float("inf")
    calls, lib = [], N.lib()
    spy = type("Spy", (), {"__getattr__": lambda self, name: (calls.append(name), getattr(lib, name))[1]})()
    outs = []
    for suits in (1, 0):
        x.grad = None
        calls.clear()
        spy.__dict__["tf24_linear16_suits"] = lambda *a, suits=suits: suits
        monkeypatch.setattr(N, "lib", lambda: spy)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = layer(x)
        y.backward(dy.transpose(0, 1).contiguous().transpose(0, 1) if suits else dy)
        monkeypatch.undo()
        assert calls.count("tf24_linear16") == (2 if suits else 0)
        outs.append((y.detach().double(), x.grad.double()))
    weight = layer.get_sparse_weights().detach().bfloat16().double().abs()
    for got, want, size, terms in ((outs[0][0], outs[1][0], x.detach().bfloat16().double().abs() @ weight.t().contiguous() + layer.bias.detach().double().abs(), k + 1),
                                   (outs[0][1], outs[1][1], dy.double().abs() @ weight, rows)):
        assert got.isnan().equal(want.isnan()) and got.isinf().equal(want.isinf())
        ok = want.isfinite()
        limit = want.abs() * 2.0 ** -7 + 2 * size * terms * 2.0 ** -23 + 1e-7
        assert ((got - want).abs() <= limit)[ok].all()


def test_dense_linear_refuses_what_it_does_not_take(cuda):
    from sparse import _native as N
    t = torch.zeros(512, 512, dtype=torch.float16, device=cuda)
    lib, p = N.lib(), t.data_ptr()
    good = dict(w=p, ldw=512, strided=0, x=p, ldx=512, dtype=N.dtype_code(torch.float16), rows=256, k=256, tokens=64, y=p, ldy=512, bias=None)
    for bad in (dict(dtype=N.dtype_code(torch.float32)), dict(rows=252), dict(rows=0), dict(k=192), dict(k=288), dict(tokens=0), dict(ldw=248), dict(ldx=252),
                dict(ldx=516), dict(ldy=248), dict(ldw=(1 << 22) + 8), dict(strided=1, ldw=248), dict(w=None), dict(x=p + 2), dict(y=p + 8), dict(bias=p + 1)):
        assert lib.tf24_linear16(*{**good, **bad}.values(), N.stream_ptr()) != 0, bad
    for shape in ((252, 256, 64), (256, 192, 64), (256, 256, 0), (0, 256, 64)):
        assert lib.tf24_linear16_suits(*shape) == 0


MANY_LONG = [(12289, 3072, 768), (1024, 3072, 2304), (1087, 3080, 2000), (2100, 1992, 3072)]          # (test_tile_rules.py)


@pytest.mark.parametrize("tokens,m,n", MANY_LONG)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_grad_weight_kernel_on_many_long_tiles(cuda, tokens, m, n, dtype):
    """The products whose 192 x 192 tiles take stages of 64 tokens: last stages of 1, 64, 63 and 52 tokens, in four pieces and in one.  Bounds
    as in the tests of the others."""
    test_grad_weight_kernel(cuda, tokens, m, n, dtype)
    test_grad_weight_kernel_is_exact_and_deterministic(cuda, tokens, m, n, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,weight_dtype,sums_dtype", [(torch.float16, torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16, None),
                                                           (torch.float16, torch.float16, None)])
@pytest.mark.parametrize("tokens,m,n", [(64, 32, 72), (64, 96, 200), (192, 3072, 768),            # one piece, the general kernel; one piece
                                        (2048, 768, 1024), (12288, 768, 72), (4096, 224, 136)])    # several: square tiles, partial ones, few columns
def test_weight_and_bias_gradient_in_one_call(cuda, dtype, weight_dtype, sums_dtype, tokens, m, n):
    """The weight's and the bias's gradient by one call of the library are, bit for bit, those of the conversion with row sums and the
    product with its result, also from pitched views; and the generator moves on alike."""
    import sparse
    from sparse.semi_structured import _mvue_weight_gradient, _spmm
    g = torch.Generator(device=cuda).manual_seed(tokens + m + n)
    grad = torch.randn(tokens, m + 8, device=cuda, generator=g).to(dtype)
    x = torch.randn(tokens, n + 16, device=cuda, generator=g).to(dtype)
    for dy, at in ((grad[:, :m], x[:, :n]), (grad[:, :m].contiguous(), x[:, 8:n + 8].contiguous())):
        torch.manual_seed(7)
        s, sums = sparse.to_sparse_semi_structured_with_row_sums(dy.t(), MVUE24=True, dtype=dtype, sums_dtype=sums_dtype)
        want = _spmm(s, at, True, out_dtype=weight_dtype)
        after = torch.cuda.default_generators[torch.cuda.current_device()].get_offset()
        torch.manual_seed(7)
        dw, db = _mvue_weight_gradient(dy, at, weight_dtype, sums_dtype)
        assert dw.dtype == weight_dtype and dw.equal(want) and db.dtype == sums.dtype and db.equal(sums)
        assert torch.cuda.default_generators[torch.cuda.current_device()].get_offset() == after


@pytest.mark.gpu
def test_weight_gradient_in_one_call_is_left_to_the_two(cuda):
    """Operands that the two calls bring into another form first, refuse or run on other kernels."""
    from sparse.semi_structured import _mvue_weight_gradient
    y, x = torch.zeros(128, 64, device=cuda, dtype=torch.float16), torch.zeros(128, 128, device=cuda, dtype=torch.float16)
    assert _mvue_weight_gradient(y, x, torch.float32, None) is not None
    for dy, at in ((y[:96], x[:96]), (y[:, :48], x), (y, x[:, :64]), (y, x[:, :100]), (y, x[:64]), (y.t().contiguous().t(), x), (y, x.t().contiguous().t()),
                   (y.float(), x.float()), (y.bfloat16(), x), (y, torch.zeros(128, 132, device=cuda, dtype=torch.float16)[:, :128]),
                   (torch.zeros(128 * 64 + 1, device=cuda, dtype=torch.float16)[1:].view(128, 64), x), (torch.nn.Parameter(y), x)):
        assert _mvue_weight_gradient(dy, at, torch.float32, None) is None
