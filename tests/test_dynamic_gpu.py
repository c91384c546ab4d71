"""Calls that take the abs-max of a tensor themselves (no accumulator, maxima of parts folded by the
consumer) against the accumulating reduction and the calibrated kernels; bit for bit."""

import pytest
import torch

from modelopt_amd import _hip
from modelopt_amd.torch.quantization.config import QuantizerAttributeConfig
from modelopt_amd.torch.quantization.nn import TensorQuantizer
from modelopt_amd.torch.quantization.qtensor import NVFP4QTensor

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = [torch.bfloat16, torch.float16, torch.float32]
# one element, a tail only, one chunk and a tail, a part, one past a part, the largest single-round
# size and one past it (1024 parts of 1024 chunks), several rounds a part
SIZES = [1, 7, 13, 8192, 8193, 8 << 20, (8 << 20) + 8 * 3 + 5, 3 * (8 << 20) + 9]


def _bits(t):
    t = t.contiguous()
    return t.view({1: torch.uint8, 2: torch.int16, 4: torch.int32}[t.element_size()])


def _tensor(n, dtype, where=-1):
    x = torch.randn(n, generator=torch.Generator(DEV).manual_seed(n), device=DEV).to(dtype)
    x[where] = -9.0
    return x


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n", SIZES)
def test_absmax_of_a_tensor(dtype, n):
    for where in (0, n // 2, n - 1):
        x = _tensor(n, dtype, where)
        for out in (dtype, torch.float32):
            assert float(_hip.absmax_tensor(x, out)) == 9.0
    x[n // 3] = float("nan")
    assert torch.isnan(_hip.absmax_tensor(x, torch.float32))
    assert _hip.absmax_tensor(x[:0], dtype) is None
    if n > 1:
        assert _hip.absmax_tensor(x[1:], dtype) is None   # unaligned: the accumulator's path


FORMATS = {
    "int8": {"num_bits": 8}, "uint4": {"num_bits": 4, "unsigned": True}, "fp8": {"num_bits": (4, 3)},
    "nvfp4": {"num_bits": (2, 1), "block_sizes": {-1: 16, "type": "dynamic", "scale_bits": (4, 3)}},
    "nvfp4_32": {"num_bits": (2, 1), "block_sizes": {-1: 32, "type": "dynamic", "scale_bits": (4, 3)}},
}


@pytest.mark.parametrize("name", FORMATS)
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", [(1, 1), (3, 7), (129, 64), (1025, 8200), (2, 65, 72)])
def test_a_dynamic_quantizer_equals_a_calibrated_one(name, dtype, shape):
    dynamic, calibrated = (TensorQuantizer(QuantizerAttributeConfig(**FORMATS[name])) for _ in range(2))
    n = 1
    for d in shape:
        n *= d
    x = _tensor(n + 1, dtype)[:n].view(shape)
    for t in (x, x.transpose(0, -1), _tensor(n + 1, dtype, 0)[1:].view(shape)):   # plain, strided, unaligned
        calibrated.reset_amax()
        calibrated.amax = t.abs().amax()
        assert torch.equal(_bits(dynamic(t)), _bits(calibrated(t)))
    grad_in = x.clone().requires_grad_()
    assert torch.equal(_bits(dynamic(grad_in).detach()), _bits(dynamic(x)))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("block", [8, 16, 32])
@pytest.mark.parametrize("shape", [(1, 32), (5, 17), (1031, 8192)])
def test_nvfp4_pack_without_a_global_scale(dtype, block, shape):
    x = _tensor(shape[0] * shape[1], dtype).view(shape)
    packed, scale, scale2 = NVFP4QTensor.quantize(x, block)
    want = _hip.nvfp4_quantize(x, x.abs().amax().float().reshape(1), block)
    for a, b in zip((packed._quantized_data, scale, scale2), want):
        assert torch.equal(_bits(a), _bits(b))


def test_under_capture_and_on_two_streams():
    x = _tensor(1 << 20, torch.bfloat16).view(1024, 1024)
    q = TensorQuantizer(QuantizerAttributeConfig(num_bits=(4, 3)))
    side = torch.cuda.Stream()
    with torch.no_grad():
        want = [q(x), q(x * 3)]
        q(x)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = q(x)
        first = x.clone()
        for i in range(4):
            x.copy_(first if i % 2 == 0 else first * 3)
            with torch.cuda.stream(side):
                other = q(first)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want[i % 2]) and torch.equal(other, want[0])
