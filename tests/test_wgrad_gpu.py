"""The masked weight gradient in one pass: the kernel against float64 products, the layer against the
separate quantizer and linear functions."""

import pytest
import torch
import torch.nn.functional as F

from modelopt_amd import _hip
from modelopt_amd.torch.quantization.config import QuantizerAttributeConfig
from modelopt_amd.torch.quantization.nn import QuantLinear
from modelopt_amd.torch.quantization.tensor_quant import MaskedGradientLinear

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = [torch.bfloat16, torch.float16]


@pytest.mark.parametrize("dtype", DTYPES)
# one token and one chunk; tokens below, at and past an octet and a step; widths with part of a
# tile; a last group of fewer than eight n tiles; several groups; below and at the kernel for many tokens, a last step of
# 31 tokens and of 8
@pytest.mark.parametrize("tokens,n,k", [(1, 8, 8), (7, 24, 136), (8, 128, 128), (64, 136, 264), (65, 1032, 128),
                                        (200, 520, 392), (513, 1160, 256),
                                        (383, 136, 392), (384, 1160, 136), (415, 24, 264), (1000, 520, 1032)])
@pytest.mark.parametrize("inner", ["all", "row", 8])
def test_kernel_against_float64(dtype, tokens, n, k, inner):
    g = torch.Generator(DEV).manual_seed(tokens)
    dy, x, w = (torch.randn(s, device=DEV, generator=g).to(dtype) for s in ((tokens, n), (tokens, k), (n, k)))
    w[0, 0], w[-1, -1], w[0, -1] = float("nan"), float("inf"), -0.0
    inner = {"all": 0, "row": k}.get(inner, inner)
    amax = 0.5 + torch.rand(w.numel() // inner if inner else 1, device=DEV, generator=g)
    amax[0] = float("nan") if inner == 8 else amax[0]
    got = _hip.wgrad_masked(dy, x, w, amax, inner)
    mask = (w.float().abs().view(amax.numel(), -1) <= amax.view(-1, 1)).view(n, k)
    exact = dy.double().t() @ x.double()
    assert torch.equal(got[~mask], torch.zeros_like(got[~mask]))
    # one rounding to the type (half a step of 7 or 10 stored bits: 2^-8, 2^-11) and fp32 sums of `tokens` products (2^-24 each, of the sum of
    # their magnitudes)
    step = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    bound = step * 1.01 * exact.abs() + tokens * 2.0 ** -24 * (dy.double().abs().t() @ x.double().abs()) + 2.0 ** -25
    assert ((got.double() - exact).abs() <= bound)[mask].all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("narrow", [False, True])
@pytest.mark.parametrize("tokens", [8, 384])
def test_the_mask_of_every_value(dtype, narrow, tokens):
    """All 65536 values of the weight under amax values between, at and beyond those of its type."""
    values = torch.arange(1 << 16, device=DEV).to(torch.uint16).view(dtype).view(1, -1)
    amax = torch.tensor([0.0, -0.0, -1.0, float("inf"), float("nan"), 1 + 2.0 ** -12, 1 - 2.0 ** -13, 9e4, 3e-8, 1e-40, -1e-9,
                         0.75, 3.4e38, 65504.0, 65519.9, 6e-5], device=DEV)
    w = values.repeat(amax.numel(), 1)
    dy, x = torch.ones(tokens, w.shape[0], device=DEV, dtype=dtype), torch.ones(tokens, w.shape[1], device=DEV, dtype=dtype)
    got = _hip.wgrad_masked(dy, x, w, amax, w.shape[1], narrow)
    limit = amax.to(dtype).float() if narrow else amax
    assert torch.equal(got, torch.where(w.float().abs() <= limit.view(-1, 1), float(tokens), 0.0).to(dtype))


def test_a_token_past_the_end_does_not_count():
    """The rows behind the last token hold NaN and infinity."""
    rows = torch.full((128, 64), float("nan"), device=DEV, dtype=torch.bfloat16)
    rows[:5] = 1.0
    w, amax = torch.zeros(64, 64, device=DEV, dtype=torch.bfloat16), torch.ones(1, device=DEV)
    assert torch.equal(_hip.wgrad_masked(rows[:5], rows[:5], w, amax), torch.full_like(w, 5.0))


WEIGHTS = {
    "int8_row": ({"num_bits": 8, "axis": 0}, lambda w: 0.8 * w.abs().amax(1, keepdim=True)),
    "int8": ({"num_bits": 8}, lambda w: 0.8 * w.abs().amax().float()),
    "fp8": ({"num_bits": (4, 3)}, lambda w: 0.8 * w.abs().amax()),
    "int4_block": ({"num_bits": 4, "block_sizes": {-1: 32, "type": "static"}},
                   lambda w: 0.8 * w.reshape(-1, 32).abs().amax(1, keepdim=True)),
    "nvfp4": ({"num_bits": (2, 1), "block_sizes": {-1: 16, "type": "dynamic", "scale_bits": (4, 3)}},
              lambda w: 0.8 * w.abs().amax()),
}


def _layer(name, dtype, bias=True):
    attributes, amax = WEIGHTS[name]
    torch.manual_seed(5)
    layer = QuantLinear(96, 136, bias=bias, device=DEV, dtype=dtype,
                        quant_desc_input=QuantizerAttributeConfig(enable=False),
                        quant_desc_weight=QuantizerAttributeConfig(**attributes))
    layer.weight_quantizer.amax = amax(layer.weight.data)
    return layer


def _separate(layer, x):
    return F.linear(x, layer.weight_quantizer(layer.weight), layer.bias)


def _grads(layer, x, y, dy, **kwargs):
    wanted = [t for t in (x, layer.weight, layer.bias) if t is not None and t.requires_grad]
    return torch.autograd.grad(y, wanted, dy, **kwargs)


@pytest.mark.parametrize("name", WEIGHTS)
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("form", ["plain", "3d", "no_bias", "input_without_gradient", "strided"])
def test_layer_equals_the_separate_functions(name, dtype, form):
    layer = _layer(name, dtype, bias=form != "no_bias")
    x = torch.randn((2, 40, 96) if form == "3d" else (80, 96), device=DEV, dtype=dtype)
    x = (x.t().contiguous().t() if form == "strided" else x).requires_grad_(form != "input_without_gradient")
    y, want_y = layer(x), _separate(layer, x)
    assert isinstance(y.grad_fn, MaskedGradientLinear._backward_cls) and torch.equal(y, want_y)
    dy = torch.randn_like(y)
    dy = dy.t().contiguous().t() if form == "strided" else dy
    for got, want in zip(_grads(layer, x, y, dy), _grads(layer, x, want_y, dy), strict=True):
        assert got.shape == want.shape and torch.equal(got == 0, want == 0)
        # the same fp32 sums in another order, each rounded to the type once: a step of it apart
        torch.testing.assert_close(got, want, rtol=2.0 ** (-7 if dtype == torch.bfloat16 else -10), atol=1e-3)


@pytest.mark.parametrize("name", ["int8_row", "int4_block", "fp8"])
def test_second_derivatives_and_batched_gradients(name):
    layer = _layer(name, torch.bfloat16)
    x = torch.randn(80, 96, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    dy = torch.randn(80, 136, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    seconds = []
    for y in (layer(x), _separate(layer, x)):
        first = _grads(layer, x, y, dy, create_graph=True)
        seconds.append(torch.autograd.grad(sum((g.float() ** 2).sum() for g in first[:2]), (x, layer.weight, dy)))
    for got, want in zip(*seconds):
        torch.testing.assert_close(got, want, rtol=2e-2, atol=2e-2 * float(want.abs().max()))
    many = torch.randn(3, 80, 136, device=DEV, dtype=torch.bfloat16)
    rows = _grads(layer, x, layer(x), many, is_grads_batched=True)
    for i in range(3):
        for got, want in zip(rows, _grads(layer, x, _separate(layer, x), many[i])):
            torch.testing.assert_close(got[i], want, rtol=2.0 ** -6, atol=2.0 ** -6 * float(want.abs().max()))


def test_what_does_not_take_it():
    layer = _layer("int8_row", torch.bfloat16)
    x = torch.randn(80, 96, device=DEV, dtype=torch.bfloat16)
    direct = MaskedGradientLinear._backward_cls
    assert isinstance(layer(x).grad_fn, direct)
    with torch.autocast("cuda", torch.float16):
        assert not isinstance(layer(x).grad_fn, direct)
    seen = []
    handle = layer.weight_quantizer.register_forward_hook(lambda m, i, o: seen.append(o.requires_grad))
    assert not isinstance(layer(x).grad_fn, direct) and seen == [True]
    handle.remove()
    layer.weight_quantizer._pass_through_bwd = True
    assert not isinstance(layer(x).grad_fn, direct)
    layer.weight_quantizer._pass_through_bwd = False
    layer.weight.requires_grad_(False)
    assert layer(x).grad_fn is None or not isinstance(layer(x).grad_fn, direct)
    with torch.no_grad():
        assert layer(x).grad_fn is None
    assert _hip.wgrad_masked(x, x[:, :60].contiguous(), x.new_zeros(96, 60), x.new_ones(1)) is None   # 60 columns


@pytest.mark.parametrize("dtype", DTYPES)
# one token and one chunk; tokens at and past a tile; n below, at and past a step, in several runs, an odd number of
# steps a run; columns with part of a tile
@pytest.mark.parametrize("tokens,n,k", [(1, 8, 8), (64, 64, 128), (65, 72, 136), (129, 1160, 264), (200, 4104, 520),
                                        (257, 2056, 4096), (512, 520, 4104), (700, 14336, 1024), (31, 4096, 1 << 16)])
def test_input_gradient_against_float64(dtype, tokens, n, k):
    g = torch.Generator(DEV).manual_seed(tokens)
    dy, w = (torch.randn(s, device=DEV, generator=g).to(dtype) for s in ((tokens, n), (n, k)))
    got, exact = _hip.input_grad(dy, w), dy.double() @ w.double()
    # as for the weight gradient, with sums of n products
    step = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    bound = step * 1.01 * exact.abs() + n * 2.0 ** -24 * (dy.double().abs() @ w.double().abs()) + 2.0 ** -25
    assert got.shape == exact.shape and ((got.double() - exact).abs() <= bound).all()
    assert torch.equal(got, _hip.input_grad(dy, w))
    dy[0, n // 2] = float("nan")
    got = _hip.input_grad(dy, w)
    assert torch.isnan(got[0]).all() and not torch.isnan(got[1:]).any()


@pytest.mark.parametrize("dtype", DTYPES)
# every tile, in one run and in several, with parts of a tile, of a step and of a run of steps
@pytest.mark.parametrize("tile,several,tokens,n,k", [(64, False, 129, 72, 520), (64, True, 200, 4104, 520), (128, False, 257, 520, 16392),
                                                     (128, True, 513, 4104, 2056), (256, False, 1000, 520, 8200),
                                                     (256, False, 200, 72, 32776), (256, True, 257, 4104, 3976),
                                                     (256, True, 700, 4104, 2056), (256, True, 385, 8200, 2056),
                                                     (256, True, 512, 14336, 4096)])
def test_every_tile_of_the_input_gradient(dtype, tile, several, tokens, n, k):
    _hip.load()
    assert _hip._entry["mo_input_grad_tile"](tokens, n, k) == tile
    assert (_hip._entry["mo_input_grad_splits"](tokens, n, k) > 1) == several
    test_input_gradient_against_float64(dtype, tokens, n, k)


def test_input_gradient_stays_inside_its_operands():
    """What lies around the operands is NaN: n and k end inside a step and a tile, the tokens inside a tile."""
    wide = torch.full((70 * 72 + 64,), float("nan"), device=DEV, dtype=torch.bfloat16)
    dy, w = wide[32:32 + 66 * 72].view(66, 72), torch.full_like(wide, float("nan"))[:72 * 64 + 32][:72 * 64].view(72, 64)
    dy.fill_(1.0)
    w.fill_(0.5)
    assert torch.equal(_hip.input_grad(dy, w), torch.full((66, 64), 36.0, device=DEV, dtype=torch.bfloat16))


def test_what_has_no_input_gradient_kernel():
    ones = torch.ones(8, 64, device=DEV, dtype=torch.bfloat16)
    assert _hip.input_grad(ones[:, :60].contiguous(), ones.new_ones(60, 8)) is None
    assert _hip.input_grad(ones.float(), ones.new_ones(64, 8).float()) is None
    assert _hip.input_grad(ones, ones.new_ones(64, 12)) is None
    assert _hip.input_grad(ones, ones.new_ones(8, 64).t()) is None
