"""The compiled calls (binding/launch.cpp): same arguments, errors and results as through ctypes."""

import pytest
import torch

from modelopt_amd import _hip

DEV = "cuda:0"
# host arrays, results by reference, or no pointers at all
THROUGH_CTYPES = {"mo_version", "mo_error_string", "mo_value_ranges", "mo_amax_fold", "mo_absmax_tensor_parts", "mo_absmax_multi",
                  "mo_nvfp4_quantize_multi", "mo_awq_clip_losses"}


def test_every_entry_point_has_its_call_and_its_argument_count():
    lib = _hip.load()
    assert set(_hip._entry) == set(_hip.SIGNATURES)
    for name, types in _hip.SIGNATURES.items():
        fn = _hip._entry[name]
        if name in THROUGH_CTYPES:
            assert fn is getattr(lib, name)
            continue
        for n in {0, len(types) - 1, len(types) + 1}:
            with pytest.raises(TypeError):
                fn(*[0] * n)
        with pytest.raises(TypeError):
            fn(*["x"] * len(types))


def test_statuses_and_conversions_without_a_launch():
    _hip.load()
    fn = _hip._entry["mo_mul_cols"]     # x, rows, cols, dtype, scale, scale dtype, y, stream
    assert fn(None, 0, 0, True, None, True, None, None) == 0
    assert fn(None, -1, 0, 2, None, 0, None, None) == _hip.MO_ERR_ARG
    assert fn(None, 1 << 40, 8, 7, None, 0, None, None) in (_hip.MO_ERR_ARG, _hip.MO_ERR_DTYPE)
    with pytest.raises(OverflowError):
        fn(None, 0, 0, 1 << 40, None, 0, None, None)
    with pytest.raises(RuntimeError, match="GPU memory"):
        _hip.row_qdq(torch.zeros(2, 16), None, _hip.MO_ROW_INT, 8, amax=torch.ones(1))
    with pytest.raises(RuntimeError, match="GPU memory"):
        _hip.dynamic_qdq(torch.zeros(2, 16), _hip.MO_ROW_INT, 8)


def _general(fn, *args, **kwargs):
    """The same call through the general path, which a timer takes"""
    with _hip.KernelTimer() as t:
        out = fn(*args, **kwargs)
    assert t.calls
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape,offset", [((1,), 0), ((3, 5), 1), ((7, 3, 48), 0), ((2, 4096), 8), ((33, 100), 3)])
def test_whole_calls_are_the_general_path(dtype, shape, offset):
    _hip.load()
    n = torch.Size(shape).numel()
    x = torch.randn(n + offset, device=DEV).to(dtype)[offset:].view(shape)
    amax = x.abs().amax().float()
    scale = torch.rand(shape[-1], device=DEV).to(dtype)
    for pre in (None, scale):
        for kind, p, a in ((_hip.MO_ROW_INT, (8, 0, 1), amax), (_hip.MO_ROW_FP8, (1, 0, 0), amax.to(dtype)),
                           (_hip.MO_ROW_NVFP4, (16, 0, 0), amax), (_hip.MO_ROW_MX, (32, 0, 0), None)):
            want = _general(_hip.row_qdq, x, pre, kind, *p, a)
            got = _hip.row_qdq(x, pre, kind, *p, a)
            assert got.dtype == dtype and got.shape == x.shape and torch.equal(got, want)
    with _hip.KernelTimer():
        want = _hip.dynamic_qdq(x, _hip.MO_ROW_INT, 8)
    got = _hip.dynamic_qdq(x, _hip.MO_ROW_INT, 8)
    assert (got is None) == (want is None) == bool(x.data_ptr() % 16)
    assert got is None or torch.equal(got, want)


@pytest.mark.gpu
def test_whole_calls_refuse_what_the_general_path_refuses():
    _hip.load()
    x = torch.randn(8, 64, device=DEV)
    amax = x.abs().amax()
    for fn in (_hip.row_qdq, lambda *a, **k: _general(_hip.row_qdq, *a, **k)):
        with pytest.raises(AssertionError):
            fn(x.t(), None, _hip.MO_ROW_INT, 8, amax=amax)
        with pytest.raises(AssertionError):
            fn(x, torch.ones(32, device=DEV), _hip.MO_ROW_INT, 8, amax=amax)
        with pytest.raises(TypeError):
            fn(x.double(), None, _hip.MO_ROW_INT, 8, amax=amax)
        with pytest.raises(RuntimeError, match="mo_row_qdq failed"):
            fn(x, None, _hip.MO_ROW_INT, 99, amax=amax)
        with pytest.raises(RuntimeError, match="GPU memory"):
            fn(x, None, _hip.MO_ROW_INT, 8, amax=amax.cpu())
    assert _hip.row_qdq(x[:0], None, _hip.MO_ROW_INT, 8, amax=amax).shape == (0, 64)
    assert _hip.dynamic_qdq(x[:0], _hip.MO_ROW_INT, 8) is None
    # a kernel and its output on the caller's stream
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        y = _hip.row_qdq(x * 2, None, _hip.MO_ROW_INT, 8, amax=amax * 2)
    s.synchronize()
    assert torch.equal(y, 2 * _hip.row_qdq(x, None, _hip.MO_ROW_INT, 8, amax=amax))
