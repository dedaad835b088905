"""The calls by which a program uses this framework, as cases that can be timed.

Each kind of case below is one thing that a user's program has the package do, through its public names:

  linear     inference: torch.nn.functional.linear of activations with a 2:4 weight, from one token to a whole prompt
  ste_fp8    the float8 layer with its weight pruned anew: soft threshold, MVUE24 compression, product
  train      one optimizer step of an MLP of two SparseLinearTranspose layers (forward, backward, masked decay, AdamW)
  s_ste      forward and backward of an MLP of two SoftThresholdLinear layers (the S-STE recipe) under autocast
  export     a trained weight pruned by magnitude and written out: compressed values, metadata, dense form
  mask       a mask refresh outside a layer: transposable search on a weight, masked decay of its gradient
  optimizer  MaskedDecayAdamW over the MLP weights and biases of a whole model
  geglu      the gated activation between the two matrices of an MLP, forward and backward

The sizes are those of the repository's benchmark and tests -- the MLP of GPT-2 (768 -> 3072 -> 768), the 11008 x 4096
weight and its transpose, 8192 x 8192 matrices -- and, for drawn cases, the ranges around them.
"""
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "2by4-pretrain_amd"))         # the package of the tree this runs in
import sparse  # noqa: E402

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32, "e4m3": torch.float8_e4m3fn}


def listed():
    return [
        # one token of one sequence against a large weight: what generating text consists of
        {"name": "decode_one_token", "kind": "linear", "tokens": 1, "n": 11008, "k": 4096, "dtype": "fp16", "bias": False},
        # a step of a batch of 37 sequences through a small layer with a bias: host work and launches count
        {"name": "decode_batch_small_layer", "kind": "linear", "tokens": 37, "n": 3072, "k": 768, "dtype": "bf16", "bias": True},
        # a prompt of a length that is no multiple of anything
        {"name": "prompt_ragged", "kind": "linear", "tokens": 3001, "n": 4096, "k": 11008, "dtype": "bf16", "bias": False},
        # the product that the benchmark's headline is taken on: a large batch of prompts
        {"name": "prompt_large", "kind": "linear", "tokens": 8192, "n": 11008, "k": 4096, "dtype": "fp16", "bias": False},
        # float8: the weight is pruned again for every product, as training in this type does (the largest case)
        {"name": "ste_fp8_layer", "kind": "ste_fp8", "tokens": 16384, "n": 8192, "k": 8192},
        # one sequence per step, masked decay and optimizer as two calls (the recipe as it is written down)
        {"name": "train_step_one_sequence", "kind": "train", "tokens": 1024, "d": 768, "hidden": 3072, "bias": True, "optimizer": "masked_add"},
        # a full batch, 12 sequences of 1024, the decay folded into the optimizer
        {"name": "train_step", "kind": "train", "tokens": 12288, "d": 768, "hidden": 3072, "bias": True, "optimizer": "masked_decay_adamw"},
        # the S-STE recipe on the same model and batch
        {"name": "s_ste_step", "kind": "s_ste", "tokens": 12288, "d": 768, "hidden": 3072, "bias": True, "dtype": "bf16"},
        # a large trained weight to its sparse form
        {"name": "export_weight", "kind": "export", "m": 8192, "k": 8192, "dtype": "bf16", "to": "fp16"},
        # every 40th optimizer step, on a float32 master weight
        {"name": "mask_refresh", "kind": "mask", "m": 11008, "k": 4096, "dtype": "fp32"},
        # the optimizer step of a 12-layer model (24 weights, 24 biases)
        {"name": "optimizer_step", "kind": "optimizer", "layers": 12, "d": 768},
        # GEGLU on a full batch
        {"name": "geglu", "kind": "geglu", "batch": 12, "seq": 1024, "hidden": 4096, "dtype": "fp16"},
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _multiple(rng, lo, hi, of):
    """A multiple of `of`, spread over the logarithm of [lo, hi]."""
    return max(of, _log(rng, lo, hi) // of * of)


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "ste_fp8", "train", "train", "s_ste", "export", "mask", "optimizer", "geglu"])
    if kind == "linear":
        if rng.random() < 0.5:
            n, k = rng.choice([(768, 768), (2304, 768), (3072, 768), (768, 3072), (4096, 4096), (11008, 4096), (4096, 11008), (8192, 8192)])
        else:                                                      # any size the compressed form takes
            n, k = _multiple(rng, 256, 12288, 32), _multiple(rng, 256, 11008, 64)
        return {"kind": kind, "tokens": _log(rng, 1, 8192), "n": n, "k": k, "dtype": rng.choice(["fp16", "bf16"]), "bias": rng.random() < 0.5}
    if kind == "ste_fp8":
        return {"kind": kind, "tokens": _log(rng, 1024, 16384), "n": _multiple(rng, 1024, 8192, 128), "k": _multiple(rng, 1024, 8192, 128)}
    if kind in ("train", "s_ste"):
        d = rng.choice([512, 640, 768, 1024, 1280, 1600])
        most = 12288 * 768 * 768 // (d * d)                        # no more work than the listed step
        if kind == "train":                                        # (the token axis of dW is compressed: multiples of 64)
            return {"kind": kind, "tokens": _multiple(rng, 512, min(16384, most), 64), "d": d, "hidden": 4 * d, "bias": rng.random() < 0.75,
                    "optimizer": rng.choice(["masked_add", "masked_decay_adamw"])}
        return {"kind": kind, "tokens": _log(rng, 500, min(16384, most)), "d": d, "hidden": 4 * d, "bias": rng.random() < 0.75,
                "dtype": rng.choice(["fp16", "bf16"])}
    if kind == "export":
        dtype, to = rng.choice([("bf16", "fp16"), ("bf16", "bf16"), ("fp16", "fp16"), ("fp32", "fp16"), ("fp32", "bf16"), ("bf16", "e4m3")])
        return {"kind": kind, "m": _multiple(rng, 768, 8192, 32), "k": _multiple(rng, 768, 8192, 128), "dtype": dtype, "to": to}
    if kind == "mask":
        return {"kind": kind, "m": _multiple(rng, 768, 11008, 32), "k": _multiple(rng, 768, 4096, 64), "dtype": rng.choice(["fp32", "bf16", "fp16"])}
    if kind == "optimizer":
        d = 64 * rng.randint(4, 12)
        return {"kind": kind, "layers": rng.randint(2, 12), "d": d}
    return {"kind": kind, "batch": rng.randint(1, 12), "seq": _log(rng, 64, 1024), "hidden": _multiple(rng, 1024, 4096, 8),
            "dtype": rng.choice(["fp16", "bf16"])}


# ------------------------------------------------------------------ what a program holds before the call
def _normal(gen, *shape, std=1.0, dtype=torch.float32):
    t = torch.randn(*shape, device="cuda", generator=gen)
    return (t * std if std != 1.0 else t).to(dtype)


def _mlp(gen, layer, case):
    """Two layers d -> hidden -> d with N(0, 0.02) weights drawn from `gen`."""
    d, h = case["d"], case["hidden"]
    layers = [layer(d, h, bias=case["bias"], device="cuda"), layer(h, d, bias=case["bias"], device="cuda")]
    with torch.no_grad():
        for m in layers:
            m.weight.normal_(std=0.02, generator=gen)
            if m.bias is not None:
                m.bias.normal_(std=0.02, generator=gen)
    return layers


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    torch.manual_seed(seed)                                        # MVUE24 draws from torch's own generator
    kind = case["kind"]
    state = {"case": case}
    if kind == "linear":
        dtype = _DTYPES[case["dtype"]]
        weight = _normal(gen, case["n"], case["k"], std=0.02, dtype=dtype)
        state["weight"] = sparse.to_sparse_semi_structured(weight, dtype=dtype)
        state["bias"] = _normal(gen, case["n"], std=0.02, dtype=dtype) if case["bias"] else None
        state["x"] = _normal(gen, 1, case["tokens"], case["k"], dtype=dtype)
    elif kind == "ste_fp8":
        x, w = _normal(gen, case["tokens"], case["k"]), _normal(gen, case["n"], case["k"], dtype=torch.bfloat16)
        in_scale, w_scale = 448.0 / x.abs().max().item(), 224.0 / w.abs().max().item()
        state["x"] = (x * in_scale).to(torch.float8_e4m3fn)
        state["w"] = w * w_scale                                   # MVUE24 rescales kept values by up to 2
        state["scale"] = 1.0 / (in_scale * w_scale)
    elif kind == "train":
        layers = _mlp(gen, sparse.SparseLinearTranspose, case)
        params = [p for m in layers for p in m.parameters()]
        if case["optimizer"] == "masked_add":
            state["opt"] = torch.optim.AdamW(params, lr=1e-4, weight_decay=0.0, fused=True)
        else:
            state["opt"] = sparse.MaskedDecayAdamW(params, lr=1e-4, weight_decay=0.0, alpha=2e-4)
        state["layers"], state["params"] = layers, params
        state["x"] = _normal(gen, case["tokens"], case["d"], dtype=torch.float16).requires_grad_()
        state["dy"] = _normal(gen, case["tokens"], case["d"], std=1e-2, dtype=torch.float16)
    elif kind == "s_ste":
        layers = _mlp(gen, sparse.SoftThresholdLinear, case)
        for m in layers:
            m.init_scale()
        state["layers"], state["params"] = layers, [p for m in layers for p in m.parameters()]
        state["dtype"] = _DTYPES[case["dtype"]]
        state["x"] = _normal(gen, case["tokens"], case["d"], dtype=state["dtype"]).requires_grad_()
        state["dy"] = _normal(gen, case["tokens"], case["d"], std=1e-2, dtype=state["dtype"])
    elif kind == "export":
        state["w"] = _normal(gen, case["m"], case["k"], dtype=_DTYPES[case["dtype"]])
        state["to"] = _DTYPES[case["to"]]
    elif kind == "mask":
        state["w"] = _normal(gen, case["m"], case["k"], std=0.02, dtype=_DTYPES[case["dtype"]])
        state["grad"] = _normal(gen, case["m"], case["k"], std=1e-3)
        state["search"] = sparse.TransposableSparse(abs=True)
    elif kind == "optimizer":
        d, h, params = case["d"], 4 * case["d"], []
        for _ in range(case["layers"]):
            for shape in ((h, d), (h,), (d, h), (d,)):
                p = torch.nn.Parameter(_normal(gen, *shape, std=0.02))
                p.grad = _normal(gen, *shape, std=1e-3)
                if len(shape) == 2:                                # 2:4 along the rows
                    p.mask = sparse.sparse24(p.detach())[1] != 0
                    p.mode = "sparse"
                params.append(p)
        state["params"] = params
        state["opt"] = sparse.MaskedDecayAdamW(params, lr=1e-4, weight_decay=1e-2, alpha=2e-4)
    else:
        dtype = _DTYPES[case["dtype"]]
        state["x"] = _normal(gen, case["batch"], case["seq"], 2 * case["hidden"], dtype=dtype).requires_grad_()
        state["dy"] = _normal(gen, case["batch"], case["seq"], case["hidden"], dtype=dtype)
        state["act"] = sparse.GELUglu()
    return state


# ------------------------------------------------------------------ one pass
def run(state):
    kind = state["case"]["kind"]
    if kind == "linear":
        with torch.no_grad():
            return F.linear(state["x"], state["weight"], state["bias"])
    if kind == "ste_fp8":
        thresholded, mask = sparse.soft_threshold24(state["w"])
        weight = sparse.to_sparse_semi_structured(state["w"], MVUE24=True, dtype=torch.float8_e4m3fn)
        return thresholded, mask, sparse.sparse_semi_structured_linear(state["x"], weight, out_dtype=torch.bfloat16, scale=state["scale"])
    if kind == "train":
        (up, down), opt, x = state["layers"], state["opt"], state["x"]
        opt.zero_grad(set_to_none=True)
        x.grad = None
        y = down(F.gelu(up(x)))
        y.backward(state["dy"])
        if state["case"]["optimizer"] == "masked_add":
            with torch.no_grad():
                for p in state["params"]:
                    if hasattr(p, "mask") and p.mode == "sparse":
                        p.grad = p.grad.float()
                        sparse.masked_add_(p.grad.data, p.data, p.mask, alpha=2e-4)
                        p.cnt = 0
        opt.step()
        return [y.detach(), x.grad] + [p.grad for p in state["params"]] + [p.detach() for p in state["params"]]
    if kind == "s_ste":
        (up, down), x = state["layers"], state["x"]
        for p in state["params"]:
            p.grad = None
        x.grad = None
        with torch.autocast("cuda", dtype=state["dtype"]):
            y = down(F.gelu(up(x)))
        y.backward(state["dy"])
        return [y.detach(), x.grad] + [p.grad for p in state["params"]]
    if kind == "export":
        weight = sparse.to_sparse_semi_structured(state["w"], dtype=state["to"])
        return weight.values(), weight.indices(), weight.to_dense()
    if kind == "mask":
        pruned, mask = state["search"](state["w"])
        grad = state["grad"]
        sparse.masked_add_(grad, state["w"], mask, alpha=2e-4)
        return pruned, mask, grad
    if kind == "optimizer":
        state["opt"].step()
        return [p.detach() for p in state["params"]]
    x = state["x"]
    x.grad = None
    y = state["act"](x)
    y.backward(state["dy"])
    return y.detach(), x.grad


# ------------------------------------------------------------------ what a pass cannot do without
def _size(name):
    return {"fp32": 4, "fp16": 2, "bf16": 2, "e4m3": 1}[name]


def work(case):
    """Inputs read once and outputs written once; a product with a 2:4 operand counts the multiply-adds of the kept half."""
    kind = case["kind"]
    if kind == "linear":
        t, n, k = case["tokens"], case["n"], case["k"]
        return {"bytes": 2 * (t * k + t * n) + n * k * 9 // 8, "flops": t * n * k}
    if kind == "ste_fp8":
        t, n, k = case["tokens"], case["n"], case["k"]
        return {"bytes": t * k + 6 * n * k + 2 * t * n, "flops": t * n * k}
    if kind in ("train", "s_ste"):
        t, d, h = case["tokens"], case["d"], case["hidden"]
        # activations of 16 bits, each crossing memory once in either direction, and of each the gradient: x and y, the
        # hidden layer before and behind its activation, read again in the backward pass
        moved = 2 * t * (4 * d + 8 * h)
        if kind == "train":
            # weight, gradient and two moments of 32 bits, the mask
            moved += 2 * d * h * (2 * 4 + 4 + 4 * 4 + 1)
            return {"bytes": moved, "flops": 6 * t * d * h}
        # weights read, gradients written; one product of three has the 2:4 weight along its inner axis
        return {"bytes": moved + 2 * d * h * 8, "flops": 10 * t * d * h}
    if kind == "export":
        m, k, out = case["m"], case["k"], _size(case["to"])
        return {"bytes": m * k * _size(case["dtype"]) + m * k * out * 3 // 2 + m * k // 8, "flops": 0}
    if kind == "mask":
        e = _size(case["dtype"])
        return {"bytes": case["m"] * case["k"] * (2 * e + 1 + 8), "flops": 0}
    if kind == "optimizer":
        return {"bytes": case["layers"] * 8 * case["d"] * case["d"] * (7 * 4 + 1), "flops": 0}
    return {"bytes": 2 * case["batch"] * case["seq"] * case["hidden"] * 8, "flops": 0}


def tolerance(case):
    """About four times what the sums taken in another order change (products, training steps), or what the same in
    float64 differs by (optimizer, activation): a 16-bit result moves by one unit in its last place where its sum lies
    near a boundary; in a training step a group of MVUE24 here and there samples another element of a gradient that
    moved that way, which is what the largest difference allows for."""
    kind, half = case["kind"], case.get("dtype") == "fp16"
    if kind == "linear":
        return {"rel": 2e-4, "max": 4e-3} if half else {"rel": 4e-4, "max": 3e-2}
    if kind == "ste_fp8":
        return {"rel": 4e-4, "max": 3e-2}
    if kind == "train":
        return {"rel": 5e-3, "max": 0.5}
    if kind == "s_ste":
        return {"rel": 5e-4, "max": 4e-3} if half else {"rel": 1e-3, "max": 3e-2}
    if kind == "optimizer":
        return {"rel": 5e-7, "max": 1.5e-6}
    if kind == "geglu":
        return {"rel": 8.5e-4, "max": 2e-3} if half else {"rel": 7e-3, "max": 1.6e-2}
    return "exact"
