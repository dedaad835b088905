"""Which operands the S-STE layer's products and weight gradients hand to the kernels as raw pointers, and which they leave to torch's operators,
which check them: on the CPU, with a stand-in for the library that notes the calls."""
import pytest
import torch
import torch.nn.functional as F
from torch import nn

TOKENS, ROWS, K = 256, 192, 320
HERE = torch.device("cpu").index


class Library:
    """Takes every product of the sizes that tf24_linear16 takes, and computes none."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        if name == "tf24_linear16_suits":
            return lambda rows, k, tokens: int(tokens > 0 and rows % 8 == 0 and k % 64 == 0 and k >= 256)
        if name == "tf24_grad_weight_workspace_bytes":
            return lambda *sizes: 0
        return lambda *args: (self.calls.append(name), 0)[1]


@pytest.fixture
def library(monkeypatch):
    from sparse import _native as N
    lib = Library()
    monkeypatch.setattr(N, "lib", lambda: lib)
    monkeypatch.setattr(N, "stream_ptr", lambda: None)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: HERE)      # (stands for "the GPU that the tensors are on")
    return lib


def draw(*shape, device="cpu", dtype=torch.bfloat16):
    return torch.randn(shape, generator=torch.Generator().manual_seed(sum(shape))).to(device=device, dtype=dtype)


class Derived(torch.Tensor):
    pass


def test_plain_operands_take_the_kernel(library):
    from sparse.sparse_ops import _product16
    x, w = draw(2, TOKENS // 2, K), draw(ROWS, K)
    assert _product16(x, w, draw(ROWS)).shape == (2, TOKENS // 2, ROWS)
    assert _product16(x, nn.Parameter(w), None).shape == (2, TOKENS // 2, ROWS)
    assert _product16(draw(TOKENS, 384), draw(384, K), None, True).shape == (TOKENS, K)
    assert library.calls == ["tf24_linear16"] * 3


@pytest.mark.parametrize("x,weight,bias", [
    (draw(TOKENS, K), draw(ROWS, K, device="meta"), None),                      # another device
    (draw(TOKENS, K, device="meta"), draw(ROWS, K), None),
    (draw(TOKENS, K), draw(ROWS, K), draw(ROWS, device="meta")),
    (draw(TOKENS, 2 * K), draw(ROWS, K), None),                                 # sizes that divide but do not match
    (draw(TOKENS, 2, K // 2), draw(ROWS, K), None),
    (draw(TOKENS, K), draw(ROWS, K).as_subclass(Derived), None),
    (draw(TOKENS, K), draw(K), None),                                           # a vector: F.linear takes it
    (draw(TOKENS, K), draw(ROWS, K, dtype=torch.float16), None)])
def test_other_operands_of_a_product_are_left_to_torch(library, x, weight, bias):
    from sparse.sparse_ops import _product16

    def outcome(fn):
        try:
            return fn()
        except RuntimeError as error:
            return type(error)
    got, want = outcome(lambda: _product16(x, weight, bias)), outcome(lambda: F.linear(x, weight, bias))
    assert library.calls == []
    assert got.shape == want.shape if isinstance(want, torch.Tensor) else got is want


def test_products_on_another_than_the_current_gpu_are_left_to_torch(library, monkeypatch):
    from sparse.sparse_ops import _product16
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)         # (the kernels go to that one's stream)
    x, w = draw(TOKENS, K), draw(ROWS, K)
    assert _product16(x, w, None).equal(F.linear(x, w))
    assert library.calls == []


@pytest.mark.parametrize("weight", [draw(ROWS, K, device="meta"), draw(768, K), draw(256, K), draw(384, K).as_subclass(Derived)])
def test_weights_that_a_hook_unpacks_otherwise_are_left_to_torch(library, weight):
    """The backward pass takes the weight from the graph: a saved-tensor hook may give back anything.  (512 gradients of 384 would be
    768 of 256 or 256 of 768.)"""
    from sparse.sparse_ops import _linear16_backward
    dy = draw(512, 384)
    with torch.no_grad():
        try:
            got = _linear16_backward(dy, None, weight, True, False, False)[0]
            assert got.shape == torch.mm(dy, weight).shape
        except RuntimeError:
            with pytest.raises(RuntimeError):
                torch.mm(dy, weight)
    assert library.calls == []


@pytest.mark.parametrize("x,taken", [
    (draw(512, 256), True), (draw(512, 256, device="meta"), False), (draw(384, 256), False), (draw(512, 256).as_subclass(Derived), False)])
def test_activations_that_a_hook_unpacks_otherwise_are_left_to_torch(library, x, taken):
    """dW = dY^T x: an activation with fewer rows than the gradient would be read past its end."""
    from sparse.sparse_ops import _linear16_backward
    dy = draw(512, 384)
    with torch.no_grad():
        if not taken and x.shape[0] != 512:
            with pytest.raises(RuntimeError):
                _linear16_backward(dy, x, None, False, True, True)
        else:
            assert _linear16_backward(dy, x, None, False, True, True)[1].shape == (384, 256)
    assert library.calls.count("tf24_grad_weight") == int(taken)
