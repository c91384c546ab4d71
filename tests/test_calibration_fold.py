"""The end of a max calibration in one launch, accumulators cleared together, and the walk over a model's modules."""

import gc
import weakref

import pytest
import torch
from torch import nn

import modelopt_amd.torch.quantization as mtq
from modelopt_amd import _hip
from modelopt_amd.torch.quantization.calib import MaxCalibrator
from modelopt_amd.torch.quantization.calib import max as cmax
from modelopt_amd.torch.quantization.nn import TensorQuantizer
from modelopt_amd.torch.quantization.nn.modules.tensor_quantizer import calibration_pass
from modelopt_amd.torch.quantization.utils import modules_of, set_training

DEV = "cuda:0"


def test_modules_in_the_order_of_the_stock_walk():
    shared = nn.Linear(2, 2)
    model = nn.Sequential(nn.Sequential(shared, nn.ReLU()), nn.ModuleList([shared, nn.Sequential(nn.ReLU())]), shared)
    model.register_module("none", None)
    model[1][1].add_module("shared", shared)
    assert [id(m) for m in modules_of(model)] == [id(m) for m in model.modules()]

    class Lists(nn.Linear):
        def named_modules(self, *a, **k):
            yield "", self
            yield "hidden", shared

    odd = nn.Sequential(Lists(2, 2), nn.ReLU())
    assert [id(m) for m in modules_of(odd)] == [id(m) for m in odd.modules()]


def test_modules_of_a_block_whose_list_is_its_own():
    hidden = nn.Sequential(nn.ReLU())
    hidden.named_modules = lambda *a, **k: iter((("", hidden),))
    for model in (nn.Sequential(hidden, nn.ReLU()), hidden):
        assert [id(m) for m in modules_of(model)] == [id(m) for m in model.modules()]
    model.modules = lambda: iter(())
    assert modules_of(model) == []


def test_a_walk_keeps_no_module_alive():
    model = nn.Sequential(nn.Linear(2, 2), nn.ReLU())
    alive = weakref.ref(model[0])
    gc.disable()
    try:
        modules_of(model)
        set_training(model, False)
        del model
        assert alive() is None
    finally:
        gc.enable()


def test_modes_are_set_as_train_sets_them():
    class Frozen(nn.Sequential):
        def train(self, mode=True):   # a block that stays in evaluation mode
            return super().train(False)

    for make in (lambda: nn.Sequential(nn.Dropout(), nn.Sequential(nn.ReLU())),
                 lambda: nn.Sequential(nn.Dropout(), Frozen(nn.ReLU()))):
        for start, mode in ((True, False), (False, True)):
            a, b = make(), make()
            a[0].training = b[0].training = not start
            a.train(mode)
            set_training(b, mode)
            assert [m.training for m in a.modules()] == [m.training for m in b.modules()]


class _Unlisted(nn.Sequential):
    def named_modules(self, *a, **k):   # its children are in no list of modules, but have a mode
        yield "", self


class _Hidden(nn.Sequential):
    def named_children(self):           # its children keep their mode
        return iter(())


def _hidden_by_instance(*children):
    block = nn.Sequential(*children)
    block.named_children = lambda: iter(())
    return block


@pytest.mark.parametrize("block", [_Unlisted, _Hidden, _hidden_by_instance])
def test_modes_of_children_that_a_block_does_not_list(block):
    for start in (True, False):
        a, b = (nn.Sequential(nn.ReLU(), block(nn.Dropout())) for _ in range(2))
        for m in (a[0], b[0], a[1][0], b[1][0]):
            m.training = start
        a.train(not start)
        set_training(b, not start)
        assert [m.training for m in (a, a[0], a[1], a[1][0])] == [m.training for m in (b, b[0], b[1], b[1][0])]


class _Layer(nn.Module):
    def __init__(self):
        super().__init__()
        self.a, self.b = nn.Linear(64, 32), nn.Linear(32, 16)

    def forward(self, x):
        return self.b(self.a(x).relu())


def test_a_disabled_and_a_collecting_quantizer_hand_their_input_back():
    q = TensorQuantizer()
    x = torch.randn(4, 8)
    q.disable()
    assert q(x) is x and q._input_dtype == x.dtype
    q.enable(), q.enable_calib(), q.disable_quant()
    seen = []
    q._calibrator.collect = lambda t: seen.append(t)
    assert q(x) is x and seen[0] is x
    assert q(x[:0]).numel() == 0 and len(seen) == 1          # nothing to show
    q.pre_quant_scale = torch.full((8,), 2.0)
    assert torch.equal(q(x), 2 * x) and torch.equal(seen[1], 2 * x)
    q.disable()
    assert torch.equal(q(x), 2 * x)


@pytest.mark.parametrize("in_a_pass", [False, True])
def test_a_calibrator_that_is_a_module(in_a_pass):
    class Calibrator(nn.Module):
        def collect(self, x):
            self.seen = x

    q = TensorQuantizer()
    q._calibrator = Calibrator()
    q.disable_quant(), q.enable_calib()
    for x in (torch.randn(4, 8), nn.Parameter(torch.randn(4, 8))):
        if in_a_pass:
            with calibration_pass():
                assert q(x) is x
        else:
            assert q(x) is x
        assert q._calibrator.seen is x


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 48, 49, 130])
def test_folded_maxima(n):
    """Accumulators and runs of parts over the limits of a launch, against torch; a NaN is the largest."""
    _hip.load()
    g = torch.Generator().manual_seed(n)
    accs, parts, dtypes, want = [], [], [], []
    for i in range(n):
        dtype = (torch.float32, torch.float16, torch.bfloat16)[i % 3]
        value = torch.rand(1, generator=g).to(dtype).float()
        runs = [torch.rand(k, generator=g).to(dtype).float() for k in (1, 255, 256, 1024)[:i % 5]]
        if i % 7 == 6:
            runs[-1:] = [torch.full((3,), float("nan"))]
        accs.append(value.to(DEV))
        parts.append([r.view(torch.int32).to(DEV) for r in runs])
        dtypes.append(dtype)
        want.append(torch.cat([value, *runs]).max().to(dtype))
    got = _hip.amax_fold(accs, parts, dtypes)
    for i in range(n):
        assert got[i].shape == () and got[i].dtype == dtypes[i]
        assert torch.equal(got[i].cpu(), want[i]) or (got[i].isnan() and want[i].isnan()), i
        assert torch.equal(accs[i].cpu()[0], want[i].float()) or want[i].isnan()
    assert len({t.untyped_storage().data_ptr() for t in got}) == n
    if n == 1:
        assert _hip.amax_fold([accs[0].cpu()], [[]], [torch.float32]) is None
        assert _hip.amax_fold(accs, [[parts]], [torch.float32]) is None
        with pytest.raises(RuntimeError, match="mo_amax_fold"):
            _hip.amax_fold(accs, [[accs[0].view(torch.int32)] * 97], [torch.float32])


@pytest.mark.gpu
def test_calibrated_values_and_accumulators_of_their_own():
    """More calibrators than the lines of one fill; a value collected after the fold; two streams."""
    g = torch.Generator(device=DEV).manual_seed(4)
    cals = [MaxCalibrator(8, None, False) for _ in range(2 * cmax._ARENA_LINES + 3)]
    xs = [torch.randn(100 + i, device=DEV, generator=g).to((torch.bfloat16, torch.float32)[i % 2]) for i in range(len(cals))]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with calibration_pass():
        for i, (c, x) in enumerate(zip(cals, xs)):
            with torch.cuda.stream(side if i % 5 == 0 else torch.cuda.current_stream()):
                c.collect(x)
    torch.cuda.synchronize()
    cmax.fold_calibrators(cals)
    assert all(c._ready is not None for c in cals)
    cals[3].collect(xs[3] * 3)                                  # the value made by the fold is out of date
    for i, (c, x) in enumerate(zip(cals, xs)):
        want = x.abs().max() * (3 if i == 3 else 1)
        first, second = c.compute_amax(), c.compute_amax()
        assert torch.equal(first, want.to(x.dtype)) and torch.equal(second, first) and first.dtype == x.dtype
        assert first.data_ptr() != second.data_ptr() and first.shape == ()
    assert cmax._arena[0] is None                               # let go of with the pass
    model = _Layer().to(DEV).to(torch.bfloat16)
    data = torch.randn(7, 64, device=DEV, generator=g).to(torch.bfloat16)
    mtq.quantize(model, mtq.FP8_DEFAULT_CFG, lambda m: (m(data), m(2 * data)))
    assert torch.equal(model.a.input_quantizer.amax, (2 * data).abs().max())
    assert torch.equal(model.b.weight_quantizer.amax, model.b.weight.abs().max())
    assert "a.input_quantizer._amax" in model.state_dict()


@pytest.mark.gpu
def test_a_timer_lists_the_fold():
    acc = torch.ones(1, device=DEV)
    with _hip.KernelTimer() as t:
        assert _hip.amax_fold([acc, acc], [[], []], [torch.float32] * 2)[1].item() == 1
        assert _hip.amax_fold([acc.cpu()], [[]], [torch.float32]) is None
    assert t.calls == {"mo_amax_fold": 1} and t.seconds["mo_amax_fold"] > 0
