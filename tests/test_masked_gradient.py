"""The linear layer whose weight gradient is computed and masked in one pass: which calls take it and what its
backward computes, with the kernel's place taken by the tensor expression; what the shortcuts past the operators take for an
interception (no GPU needed)."""

import pytest
import torch

from modelopt_amd import _hip
from modelopt_amd.torch.quantization import kernels
from modelopt_amd.torch.quantization.nn import QuantLinear
from modelopt_amd.torch.quantization.tensor_quant import MaskedGradientLinear


@pytest.mark.parametrize("n,k,most", [
    (14336, 4096, 1024), (2048, 2048, 1024), (2048, 2040, 512), (16384, 128, 512), (512, 512, 512), (24, 4096, 512),
    (16, 4096, 512), (8, 4096, 256), (8, 1 << 20, 256), (65536, 24, 512), (65536, 16, 64), (65536, 8, 64), (1 << 20, 8, 64),
    (8, 8, 64), (12, 4096, 0), (4096, 20, 0)])
def test_the_sizes_at_which_one_pass_pays(n, k, most):
    """By the tokens up to which it was measured to be no slower than the product and the mask."""
    for tokens in (0, 1, most, most + 1, 4096):
        assert kernels.wgrad_mask_pays(tokens, n, k) == (1 <= tokens <= most), tokens


@pytest.mark.parametrize("n,k,most", [(14336, 4096, 1024), (4096, 4096, 1024), (4088, 4096, 512), (6144, 6144, 512),
                                      (6136, 6144, 256), (7168, 7168, 256), (8, 8, 1024), (8, 16384, 256), (12, 8, 0), (8, 12, 0)])
def test_the_sizes_at_which_the_input_gradient_is_left_to_the_kernel(n, k, most):
    for tokens in (0, 1, most, most + 1, 4096):
        assert kernels.input_grad_pays(tokens, n, k) == (1 <= tokens <= most), tokens


@pytest.mark.parametrize("n,k,most", [(8, 32768, 128), (53248, 32768, 128), (8192, 28672, 128), (4096, 40960, 0), (8, 32776, 0),
                                      (16384, 16384, 256), (16392, 16384, 128), (53248, 8192, 256), (53248, 8200, 128), (8, 16392, 128)])
def test_the_widest_results_that_are_left_to_the_input_gradient_kernel(n, k, most):
    for tokens in (0, 1, 128, 129, 256, 257):
        assert kernels.input_grad_pays(tokens, n, k) == (1 <= tokens <= most), tokens


def _halves(w):   # a quantizer of the CPU: to steps of a half within +-1
    return (w.clamp(-1, 1) * 2).round() / 2


@pytest.fixture
def made(monkeypatch):
    """The weight gradients that were computed."""
    done = []

    def wgrad_masked(dy, x, w, amax, inner=0, narrow_amax=False):
        done.append("weight")
        return torch.where(w.abs() <= amax.reshape(-1, 1), dy.t() @ x, torch.zeros(()))

    monkeypatch.setattr(_hip, "wgrad_masked", wgrad_masked)
    return done


def _case(leaf=True, bias=True):
    g = torch.Generator().manual_seed(3)
    x = torch.randn(5, 8, generator=g, requires_grad=True)
    w = torch.randn(16, 8, generator=g, requires_grad=True)
    b = torch.randn(16, generator=g, requires_grad=True) if bias else None
    seen = x if leaf else x * 1.0
    return x, w, b, seen, MaskedGradientLinear.apply(seen, w, b, _halves, torch.ones(()), 0)


@pytest.mark.parametrize("leaf", [True, False])
@pytest.mark.parametrize("bias", [True, False])
def test_only_the_gradients_that_are_asked_for_are_computed(made, leaf, bias):
    x, w, b, seen, y = _case(leaf, bias)
    dy = torch.randn(5, 16, generator=torch.Generator().manual_seed(4))
    products = []

    class Count(torch.utils._python_dispatch.TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            if func is torch.ops.aten.mm.default:
                products.append(tuple(args[1].shape))
            return func(*args, **(kwargs or {}))

    want = {"x": dy @ _halves(w.detach()), "w": torch.where(w.detach().abs() <= 1, dy.t() @ x.detach(), torch.zeros(())),
            "b": dy.sum(0)}
    tensors = {"x": x, "w": w, "b": b}
    for names in (("x",), ("w",), ("b",), ("x", "w"), ("w", "b"), ("x", "w", "b")):
        if b is None and "b" in names:
            continue
        made.clear()
        got = torch.autograd.grad(y, [tensors[n] for n in names], dy, retain_graph=True)
        for n, t in zip(names, got):
            assert torch.equal(t, want[n])
        assert made == (["weight"] if "w" in names else [])
        with Count():
            products.clear()
            torch.autograd.grad(y, [tensors[n] for n in names], dy, retain_graph=True)
        # [16, 8] for the input; the tensor expression of the weight's under a dispatch mode
        assert products == [(16, 8)] * ("x" in names) + [(5, 8)] * ("w" in names)
    made.clear()
    y.backward(dy, inputs=[w], retain_graph=True)
    assert made == ["weight"] and x.grad is None and torch.equal(w.grad, want["w"])
    w.grad = None
    y.backward(dy)
    assert torch.equal(x.grad, want["x"]) and torch.equal(w.grad, want["w"]) and (b is None or torch.equal(b.grad, want["b"]))


@pytest.mark.parametrize("trained_input", [True, False])
def test_the_quantised_weight_is_kept_for_the_gradient_of_the_input_only(made, trained_input):
    x = torch.randn(5, 8, requires_grad=trained_input)
    w = torch.randn(16, 8, requires_grad=True)
    kept = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(t) or t, lambda t: t):
        y = MaskedGradientLinear.apply(x, w, None, _halves, torch.ones(()), 0)
    quantized = [t for t in kept if t.shape == w.shape and t is not w and torch.equal(t, _halves(w.detach()))]
    assert len(quantized) == trained_input
    y.sum().backward()
    assert w.grad is not None and (x.grad is not None) == trained_input


def test_a_default_device_is_no_interception():
    class Follows(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    assert not kernels.torch_is_intercepted()
    with torch.device("cpu"):
        assert not kernels.torch_is_intercepted()
        with Follows():
            assert kernels.torch_is_intercepted()
    with Follows(), torch.device("meta"):
        assert kernels.torch_is_intercepted()
    torch.set_default_device("cpu")
    try:
        assert not kernels.torch_is_intercepted()
    finally:
        torch.set_default_device(None)


def test_a_compiler_does_not_follow_the_choice_of_the_route(monkeypatch):
    layer = QuantLinear(8, 8)
    for quantizer in (layer.input_quantizer, layer.weight_quantizer, layer.output_quantizer):
        quantizer.disable()
    asked = []
    monkeypatch.setattr(type(layer), "_masked_gradient_linear", lambda self, x: asked.append(x))
    x = torch.randn(4, 8)
    want = layer(x)
    assert len(asked) == 1
    monkeypatch.setattr(torch.compiler, "is_compiling", lambda: True)
    assert torch.equal(layer(x), want) and len(asked) == 1
