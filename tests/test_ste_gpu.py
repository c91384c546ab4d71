"""The clipping straight-through backward in one launch against the tensor expression it replaces."""

import pytest
import torch

from modelopt_amd import _hip
from modelopt_amd.torch.quantization import kernels
from modelopt_amd.torch.quantization.tensor_quant import _fake_tensor_quant_backward, fake_tensor_quant

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _bits(t):
    return t.view(torch.int32 if t.dtype == torch.float32 else torch.int16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
# below one chunk, tails of every kind, one tile and its edges, rows of whole and of broken chunks
@pytest.mark.parametrize("shape,amax_shape", [
    ((5,), ()), ((8192,), (1,)), ((8199,), ()), ((3, 2731), (1, 1)), ((33, 256), (33, 1)), ((7, 13), (7, 1)),
    ((4, 6, 24), (1, 6, 1)), ((64, 130), (1, 130)), ((2, 16, 2, 16), (2, 1, 2, 1))])
@pytest.mark.parametrize("amax_dtype", [torch.float32, None])
def test_mask_equals_the_tensor_expression(dtype, shape, amax_shape, amax_dtype):
    g = torch.Generator().manual_seed(3)
    x = torch.randn(shape, generator=g).to(dtype)
    grad = torch.randn(shape, generator=g).to(dtype)
    amax = (0.5 + torch.rand(amax_shape, generator=g)).to(amax_dtype or dtype)
    flat = x.view(-1)
    flat[:5] = torch.tensor([float("nan"), float("inf"), -0.0, 0.0, float("-inf")]).to(dtype)
    flat[-1] = amax.reshape(-1)[-1].to(dtype)      # on (or one rounding away from) the limit itself
    grad.view(-1)[2] = -0.0
    grad.view(-1)[3] = float("nan")
    want = torch.where(x.abs() <= amax, grad, torch.zeros(1, dtype=dtype))
    got = _fake_tensor_quant_backward(x.to(DEV), amax.to(DEV), grad.to(DEV)).cpu()
    assert got.dtype == want.dtype and torch.equal(_bits(got), _bits(want))


@pytest.mark.parametrize("limit", [float("nan"), float("inf"), 0.0, -1.0])
def test_special_limits(limit):
    x = torch.tensor([0.0, -0.0, 1.0, float("inf"), float("nan"), -2.0, 3.0, 4.0, 5.0]).bfloat16()
    grad = torch.arange(1, 10).bfloat16()
    amax = torch.tensor(limit)
    want = torch.where(x.abs() <= amax, grad, torch.zeros(1, dtype=grad.dtype))
    got = _fake_tensor_quant_backward(x.to(DEV), amax.to(DEV), grad.to(DEV)).cpu()
    assert torch.equal(_bits(got), _bits(want))


def test_unaligned_and_uncovered_inputs():
    g = torch.Generator().manual_seed(4)
    x, grad = (torch.randn(1001, generator=g).bfloat16() for _ in range(2))
    amax = torch.tensor(0.7)
    want = torch.where(x.abs() <= amax, grad, torch.zeros(1, dtype=grad.dtype))[1:]
    xd, gd = x.to(DEV)[1:], grad.to(DEV)[1:]       # two bytes off a 16-byte boundary
    assert torch.equal(_bits(_hip.ste_mask(xd, gd, amax.to(DEV).reshape(1), 1, 1, 1000, True).cpu()), _bits(want))
    # a gradient of another type or memory order takes the tensor expression
    assert kernels.ste_mask(xd, amax.to(DEV), gd.float()) is None
    m = torch.randn(8, 16, device=DEV)
    assert kernels.ste_mask(m, amax.to(DEV), torch.randn(16, 8, device=DEV).t()) is None


def test_a_gradient_that_is_differentiated_or_batched():
    """``create_graph`` and ``is_grads_batched`` see the tensor expression of the mask."""
    x = torch.linspace(-2, 2, 64, device=DEV).requires_grad_()
    amax = torch.tensor(1.0, device=DEV)
    mask = (x.detach().abs() <= 1).float()
    v = torch.randn(64, generator=torch.Generator(DEV).manual_seed(0), device=DEV, requires_grad=True)
    g, = torch.autograd.grad(fake_tensor_quant(x, amax), x, v, create_graph=True)
    again, = torch.autograd.grad(g.sum(), v)
    assert torch.equal(again, mask)
    y = fake_tensor_quant(x, amax)
    rows, = torch.autograd.grad(y, x, torch.eye(64, device=DEV), is_grads_batched=True)
    assert torch.equal(rows, torch.diag(mask))
