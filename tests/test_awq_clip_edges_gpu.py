"""The 16-bit clip search at the edges of its tiles: 32 rows (bf16) or 64 rows (fp16) per wavefront, tiles
of 32 tokens or groups of 4, passes of 64, shares of the ratios, codes too wide for the short
quotient, blocks whose scale leaves the range of the reciprocal, products that overflow."""

import pytest
import torch

from modelopt_amd import _hip
from oracle import awq as oawq
from oracle import reduce

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
RATIOS = [round(0.5 + 0.05 * i, 2) for i in range(10)] + [1.0]


def _case(n, k, tokens, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    w = (0.05 * torch.randn(n, k, generator=g)).to(dtype)
    x = (torch.randn(tokens, k, generator=g) * torch.exp(0.5 * torch.randn(1, k, generator=g))).to(dtype)
    return w, x


def _losses(w, x, block, num_bits=4, ratios=RATIOS):
    w_amax = reduce.reduce_amax(w.reshape(-1, block), axis=[1], keepdims=True)
    loss = torch.zeros(len(ratios), w.shape[0], w.shape[1] // block, device=DEV)
    assert _hip.awq_clip_losses_into(x.to(DEV), w.to(DEV), w_amax.to(DEV), ratios, block, num_bits, False, False, loss)
    return loss.cpu()


def _check(got, want):
    """Sums in another order flip the rounding of a partial output now and then (one step of the dtype
    of one token's error); the losses of a ratio agree on aggregate as in the tests of the kernel."""
    for i, r in enumerate(RATIOS):
        assert float((got[i] - want[r]).abs().sum() / want[r].abs().sum()) < 2e-4, r


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,k,tokens,block", [
    (1, 16, 1, 16), (31, 64, 31, 16), (33, 128, 32, 128), (65, 256, 33, 64), (129, 128, 63, 32), (257, 128, 66, 128),
    (130, 64, 5, 64), (64, 32, 127, 32)])
def test_tile_edges(dtype, n, k, tokens, block):
    w, x = _case(n, k, tokens, dtype, n + tokens)
    want, _ = oawq.awq_clip_search(w, [x], block, 4, max_tokens_per_batch=1 << 20)
    _check(_losses(w, x, block), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_wide_codes_and_extreme_scales(dtype):
    w, x = _case(40, 128, 20, dtype, 3)
    want, _ = oawq.awq_clip_search(w, [x], 64, 13, max_tokens_per_batch=1 << 20)
    got = _losses(w, x, 64, num_bits=13)
    for i, r in enumerate(RATIOS[:-1]):    # 13 bits: only clipping costs anything worth comparing
        assert float((got[i] - want[r]).abs().sum() / want[r].abs().sum()) < 2e-4, r
    if dtype == torch.bfloat16:            # a block below 2^-64: the divided form, exact zeros apart
        w[:, :64] *= 2.0 ** -90
        want, _ = oawq.awq_clip_search(w, [x], 64, 4, max_tokens_per_batch=1 << 20)
        _check(_losses(w, x, 64), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_shares_of_the_ratios_give_the_same_bits(dtype):
    """few rows share the ratios between wavefronts, many do not; a row's losses do not depend on it"""
    w, x = _case(4096, 1024, 40, dtype, 9)
    whole = _losses(w, x, 16)
    for r0 in (0, 1024, 4032):
        rows = slice(r0, r0 + 64)
        assert torch.equal(_losses(w[rows].contiguous(), x, 16), whole[:, rows])
        one = _losses(w[rows].contiguous(), x, 16, ratios=RATIOS[3:4])
        assert torch.equal(one[0], whole[3, rows])


# rows in the first and the last place of a tile and in the part of one at the end, tokens in the first and a
# later pass and in the part of a group at the end
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("kind", ["overflow", "clipped_overflow", "both_signs", "inf", "nan"])
@pytest.mark.parametrize("n,k,tokens,block,rows,token", [
    (96, 64, 8, 32, (21,), 3), (129, 128, 66, 128, (0, 63, 128), 65), (70, 32, 70, 16, (5, 37, 64), 31), (64, 64, 1, 64, (33,), 0)])
def test_a_row_that_is_not_finite_leaves_the_others_alone(dtype, kind, n, k, tokens, block, rows, token):
    """Products of finite values that overflow, and weights that are not finite: the losses of all other rows
    are to the bit those of the same weight without them, and the row's own are what the CPU makes of it."""
    w, x = _case(n, k, tokens, dtype, n)
    clean, col = w.clone(), k - 3
    # times 4096 past 65504, times 64 past 2^128; the last one only where clipping widens it (code -8 of 7)
    scale, x_large = (1.0, 4096.0) if dtype == torch.float16 else (2.0 ** 118, 64.0)
    values = {"overflow": (0.0, 20.0), "both_signs": (-20.0, 20.0), "clipped_overflow": (0.0, -15.875)}
    for r in rows:
        w[r, col - 1:col + 1] = torch.tensor(values[kind]) * scale if kind in values else float(kind)
        clean[r, col - 1:col + 1] = 0.0
    if kind in values:
        x[token, col - 1:col + 1] = x_large
    got, other = _losses(w, x, block), _losses(clean, x, block)
    want, _ = oawq.awq_clip_search(w, [x], block, 4, max_tokens_per_batch=1 << 20)
    healthy = torch.ones(n, dtype=torch.bool)
    healthy[list(rows)] = False
    assert torch.isfinite(other[:, healthy]).all() and torch.equal(got[:, healthy], other[:, healthy])
    assert torch.equal(got[:, :, :col // block], other[:, :, :col // block])      # the other blocks of the row
    for i, r in enumerate(RATIOS):
        mine, cpu = got[i][~healthy][:, col // block], want[r][~healthy][:, col // block]
        assert kind == "clipped_overflow" or not torch.isfinite(cpu).any()
        assert torch.equal(mine.isnan(), cpu.isnan()) and torch.equal(mine.isinf(), cpu.isinf()), r
        # what is finite and large is one token's error, above 1700: two outputs in steps of 32
        large = torch.isfinite(cpu) & (cpu * tokens > 3e6)
        torch.testing.assert_close(mine[large], cpu[large], rtol=0.08, atol=0.0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("block", [32, 64, 128])
def test_sums_are_made_in_chains_of_a_quarter_of_a_block(dtype, block):
    """One large weight at either end of a block, small ones between: 2^24 + 1 is 2^24 in fp32, so that the
    chains with the large ones lose small ones, and no other chain does.  Quantised, the small ones are zero and
    the large ones themselves: the loss is the square of what the sum of the block has kept, half of it at least."""
    w = torch.full((96, 2 * block), 2.0 ** -11).to(dtype)      # a pair of products: 2^-10
    w.view(96, 2, block)[..., 0], w.view(96, 2, block)[..., -1] = 2.0 ** 14, -2.0 ** 14
    kept = block / 2 * 2.0 ** -11
    loss = _losses(w, torch.ones(1, 2 * block).to(dtype), block, ratios=[1.0])
    assert (loss >= kept * kept).all() and (loss <= (2 * kept) ** 2).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("ratios,blocks", [(1, 1), (11, 255), (11, 257), (3, 5000)])
def test_best_clip_is_what_the_loop_over_the_ratios_leaves(dtype, ratios, blocks):
    g = torch.Generator().manual_seed(blocks)
    loss = torch.rand(ratios, blocks, generator=g).mul_(4).round_()      # many equal losses
    loss[torch.rand(ratios, blocks, generator=g) < 0.2] = float("nan")
    loss[torch.rand(ratios, blocks, generator=g) < 0.2] = float("inf")
    loss[:, 0] = float("nan")
    loss[:, -1] = float("inf") if blocks > 1 else loss[:, -1]
    amax, table = torch.rand(blocks, 1, generator=g).to(dtype), torch.linspace(0.5, 1, ratios)
    best, clip = torch.full((blocks, 1), float("inf")), torch.zeros(blocks, 1, dtype=dtype)
    for r in range(ratios):
        better = loss[r].view(-1, 1) < best
        best = torch.where(better, loss[r].view(-1, 1), best)
        clip = torch.where(better, (amax.float() * table[r]).to(dtype), clip)
    got_best, got_clip = _hip.awq_best_clip(loss.to("cuda"), table.to("cuda"), amax.to("cuda"))
    assert torch.equal(got_best.cpu(), best) and torch.equal(got_clip.cpu(), clip)
