"""Row-wise fake quantisation (pre-scaled, ragged or unaligned rows): integers and FP8 against the kernels for
whole tensors, which the oracle tests pin, NVFP4 and the MX formats, whose other entry points run the same
kernel, against the oracle; bit for bit."""

import pytest
import torch
import torch.nn.functional as F

from conftest import assert_bits_equal
from modelopt_amd import _hip
from oracle import fake_quant, mx, qtensor

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = [torch.bfloat16, torch.float16, torch.float32]
MX = {name: i for i, name in enumerate(_hip.ELEM_FORMATS[:-1])}


def _whole(x, kind, p0, p1, p2, amax):
    if kind == _hip.MO_ROW_INT:
        return _hip.int_qdq(x, amax, 1, 1, x.numel(), p0, p1, p2)
    if kind == _hip.MO_ROW_FP8:
        return _hip.fp8_qdq(x, amax, 1, 1, x.numel(), bool(p0))
    x = x.cpu()
    if kind == _hip.MO_ROW_MX:
        return mx.block_fp_fake_quant(x, p0, _hip.ELEM_FORMATS[p1])
    if p1 == 0:
        return fake_quant.nvfp4_fake_quant(x, amax.cpu(), p0)
    k = x.shape[-1]
    padded, wsf2 = F.pad(x, (0, -k % p0)), amax.cpu().float().reshape(()) / 2688.0
    packed, wsf, _ = qtensor.nvfp4_quantize(padded, p0, wsf2=wsf2)
    return qtensor.nvfp4_dequantize(packed, wsf, wsf2, p0, padded.shape, x.dtype)[..., :k]


KINDS = ([(_hip.MO_ROW_INT, 8, 0, 0), (_hip.MO_ROW_INT, 4, 1, 0), (_hip.MO_ROW_INT, 16, 0, 1),
          (_hip.MO_ROW_FP8, 1, 0, 0), (_hip.MO_ROW_FP8, 0, 0, 0)]
         + [(_hip.MO_ROW_NVFP4, b, m, 0) for b in (8, 16, 32) for m in (0, 1)]
         + [(_hip.MO_ROW_MX, b, f, 0) for b, f in zip((8, 16, 32, 8, 16, 32, 8, 16, 32), MX.values())])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind,p0,p1,p2", KINDS)
# one element, less than a chunk, one past a chunk or a block, whole blocks, tiles with a remainder
@pytest.mark.parametrize("rows,k", [(1, 1), (3, 7), (5, 17), (2, 33), (7, 64), (130, 65), (33, 1030)])
@pytest.mark.parametrize("pre", [False, True])
def test_equals_the_whole_tensor_kernels(dtype, kind, p0, p1, p2, rows, k, pre):
    g = torch.Generator().manual_seed(rows * 1000 + k)
    x = (torch.randn(rows, k, generator=g) * torch.exp(torch.randn(rows, k, generator=g))).to(dtype)
    x.view(-1)[::37] = 0.0
    x.view(-1)[1::53] = -0.0
    x = x.to(DEV)
    s = torch.exp(0.5 * torch.randn(k, generator=g)).to(dtype).to(DEV) if pre else None
    seen = x * s if pre else x
    amax = None if kind == _hip.MO_ROW_MX else (0.8 * seen.abs().amax()).float().reshape(1)
    got = _hip.row_qdq(x, s, kind, p0, p1, p2, amax)
    assert_bits_equal(got.cpu(), _whole(seen, kind, p0, p1, p2, amax).cpu().contiguous(), "qdq")


# both sides of the sizes between which a whole tensor without a scale goes to the kernel for whole tensors
@pytest.mark.parametrize("dtype,line", [(torch.float32, 1 << 22), (torch.float32, 1 << 28), (torch.float16, 1 << 20),
                                        (torch.float16, 1 << 24), (torch.bfloat16, 1 << 23), (torch.bfloat16, 1 << 24)])
@pytest.mark.parametrize("kind,p0,p1,p2", KINDS[:5])
def test_large_tensors_equal_their_parts(dtype, line, kind, p0, p1, p2):
    g = torch.Generator(DEV).manual_seed(p0)
    x = torch.randn(line + 8, device=DEV, generator=g).to(dtype)
    if dtype != torch.float32:
        x[:65536] = torch.arange(65536, device=DEV, dtype=torch.int32).to(torch.int16).view(dtype)   # every value
    x[-3], x[-2] = float("nan"), float("inf")
    amax = torch.full((1,), 2.5, device=DEV)
    step = 1 << 19
    parts = torch.cat([_hip.row_qdq(t.clone(), None, kind, p0, p1, p2, amax) for t in x.split(step)])
    for n in (line - 8, line, line + 8):
        got = _hip.row_qdq(x[:n], None, kind, p0, p1, p2, amax)
        same = (got == parts[:n]) | (torch.isnan(got) & torch.isnan(parts[:n]))
        assert bool(same.all()) and torch.equal(torch.signbit(got), torch.signbit(parts[:n]))


@pytest.mark.parametrize("kind,p0,p1,p2", [(_hip.MO_ROW_FP8, 1, 0, 0), (_hip.MO_ROW_MX, 32, 0, 0)]
                         + [(_hip.MO_ROW_NVFP4, b, m, 0) for b in (8, 16, 32) for m in (0, 1)]
                         + [(_hip.MO_ROW_MX, b, f, 0) for b, f in zip((8, 16, 32, 8, 16, 32, 8, 16), list(MX.values())[1:])])
@pytest.mark.parametrize("dtype", DTYPES)
def test_unaligned_base_and_non_finite_blocks(dtype, kind, p0, p1, p2):
    g = torch.Generator().manual_seed(1)
    flat = torch.randn(40 * 96 + 1, generator=g).to(dtype)
    flat[5], flat[700], flat[1500] = float("nan"), float("inf"), float("-inf")
    x = flat.to(DEV)[1:].view(40, 96)                 # an element off a 16-byte boundary
    amax = torch.full((1,), 3.0, device=DEV)
    got = _hip.row_qdq(x, None, kind, p0, p1, p2, None if kind == _hip.MO_ROW_MX else amax)
    assert_bits_equal(got.cpu(), _whole(x.clone(), kind, p0, p1, p2, amax).cpu(), "qdq")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("block", [8, 16, 32])
@pytest.mark.parametrize("rows,k", [(1, 3), (9, 40), (130, 72), (17, 1000)])
def test_nvfp4_quantize_of_ragged_rows_equals_padded_rows(dtype, block, rows, k):
    g = torch.Generator().manual_seed(k)
    x = torch.randn(rows, k, generator=g).to(dtype).to(DEV)
    padded = F.pad(x, (0, -k % block)).contiguous()
    amax = x.abs().amax().float()
    got, want = (_hip.nvfp4_quantize(t, amax, block) for t in (x, padded))
    for a, b in zip(got, want):
        assert torch.equal(a.view(torch.uint8) if a.dtype != torch.float32 else a,
                           b.view(torch.uint8) if b.dtype != torch.float32 else b)
    # the literal division of every element, and the scales handed in, give the same codes
    exact = _hip.nvfp4_quantize(x, amax, block, flags=_hip.MO_FLAG_FORCE_EXACT)
    given = _hip.nvfp4_quantize(x, got[2], block, True, got[1])
    assert torch.equal(exact[0], got[0]) and torch.equal(given[0], got[0])


FORMATS = {
    "int8": {"num_bits": 8}, "uint4": {"num_bits": 4, "unsigned": True}, "fp8": {"num_bits": (4, 3)},
    "nvfp4": {"num_bits": (2, 1), "block_sizes": {-1: 16, "type": "dynamic", "scale_bits": (4, 3)}},
    "mxfp6": {"num_bits": (3, 2), "block_sizes": {-1: 32, "type": "dynamic", "scale_bits": (8, 0)}},
    "mxint8": {"num_bits": 8, "block_sizes": {-1: 8, "type": "dynamic", "scale_bits": (8, 0)}},
    # two-level scales of another element format, and blocks of 64, have no one-pass form
    "e1m2": {"num_bits": (1, 2), "block_sizes": {-1: 16, "type": "dynamic", "scale_bits": (4, 3)}},
}


@pytest.mark.parametrize("name", FORMATS)
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("form", ["plain", "transposed", "unaligned", "scale_fp32", "grad", "dynamic", "collects"])
def test_a_pre_quant_scale_equals_the_scaled_input(name, dtype, form):
    from modelopt_amd.torch.quantization.config import QuantizerAttributeConfig
    from modelopt_amd.torch.quantization.nn import TensorQuantizer

    g = torch.Generator().manual_seed(3)
    flat = torch.randn(2 * 9 * 72 + 1, generator=g).mul_(3).to(dtype)
    flat[77], flat[300], flat[900] = float("nan"), float("inf"), float("-inf")
    flat = flat.to(DEV)
    x = flat[1:] if form == "unaligned" else flat[:-1]
    x = x.view(2, 72, 9).transpose(1, 2) if form == "transposed" else x.view(2, 9, 72)
    scale = torch.exp(0.5 * torch.randn(72, generator=g)).to(torch.float32 if form == "scale_fp32" else dtype).to(DEV)
    plain, scaled = (TensorQuantizer(QuantizerAttributeConfig(**FORMATS[name])) for _ in range(2))
    scaled.pre_quant_scale = scale
    if form != "dynamic" and not plain.is_mx_format:
        plain.amax = scaled.amax = torch.tensor(2.5, dtype=dtype, device=DEV)
    if form == "collects":
        plain.enable_calib(), scaled.enable_calib()
    if form == "grad":
        x = x.clone().requires_grad_()
    got, want = scaled(x), plain(x * scale)
    assert got.dtype == want.dtype and got.shape == want.shape
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    keep = ~torch.isnan(want)
    assert torch.equal(got[keep], want[keep])


FORMS = ["plain", "one_dim", "strided", "unaligned", "parameter", "scaled", "dynamic", "amax_1x1", "amax_on_cpu",
         "nan_overflow", "inference"]
# float64 is taken with a calibrated abs-max only, without blocks and scales
DIRECT = [(name, dtype, form) for name in FORMATS for dtype in DTYPES + [torch.float64] for form in FORMS
          if dtype != torch.float64 or not (FORMATS[name].get("block_sizes") or form in ("scaled", "dynamic"))]


@pytest.mark.parametrize("name,dtype,form", DIRECT)
def test_the_direct_route_equals_the_steps_of_forward(name, dtype, form, monkeypatch):
    from modelopt_amd.torch.quantization.config import QuantizerAttributeConfig
    from modelopt_amd.torch.quantization.nn import TensorQuantizer
    from modelopt_amd.torch.quantization.overflow import set_fp8_overflow_behavior

    flat = torch.randn(11 * 96 + 1, generator=torch.Generator().manual_seed(6)).mul_(3).to(dtype).to(DEV)
    x = (flat[1:] if form == "unaligned" else flat[:-1]).view(11, 96)
    x = {"one_dim": x[3], "strided": x[:, :].t().contiguous().t(), "parameter": torch.nn.Parameter(x)}.get(form, x)
    q = TensorQuantizer(QuantizerAttributeConfig(**FORMATS[name]))
    if form == "scaled":
        q.pre_quant_scale = torch.linspace(0.5, 2, 96).to(dtype).to(DEV)
    if form != "dynamic" and not q.is_mx_format:
        q.amax = torch.full((1, 1) if form == "amax_1x1" else (), 2.5, dtype=dtype,
                            device="cpu" if form == "amax_on_cpu" else DEV)
    previous = set_fp8_overflow_behavior("nan" if form == "nan_overflow" else "auto")
    try:
        with torch.inference_mode(form == "inference"), torch.no_grad():
            got = q(x)
            monkeypatch.setattr(TensorQuantizer, "_direct_fake_quant", lambda self, inputs: None)
            want = q(x)
    finally:
        set_fp8_overflow_behavior(previous)
    assert got.shape == want.shape and got.dtype == want.dtype and got.is_contiguous() == want.is_contiguous()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got.nan_to_num(nan=0.0), want.nan_to_num(nan=0.0))
