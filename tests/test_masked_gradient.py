"""The linear layer whose weight gradient is computed and masked in one pass: which calls take it and what its
backward computes, with the kernel's place taken by the tensor expression (no GPU needed)."""

import pytest

from modelopt_amd.torch.quantization import kernels


@pytest.mark.parametrize("n,k,most", [
    (14336, 4096, 1024), (2048, 2048, 1024), (2048, 2040, 512), (16384, 128, 512), (512, 512, 512), (24, 4096, 512),
    (16, 4096, 512), (8, 4096, 256), (8, 1 << 20, 256), (65536, 24, 512), (65536, 16, 64), (65536, 8, 64), (1 << 20, 8, 64),
    (8, 8, 64), (12, 4096, 0), (4096, 20, 0)])
def test_the_sizes_at_which_one_pass_pays(n, k, most):
    """By the tokens up to which it was measured to be no slower than the product and the mask."""
    for tokens in (0, 1, most, most + 1, 4096):
        assert kernels.wgrad_mask_pays(tokens, n, k) == (1 <= tokens <= most), tokens
