"""Shape logic between torch tensors and the HIP C ABI (``modelopt_amd._hip``).

Everything here runs on the GPU through ``libmodelopt_hip.so``; CPU tensors are rejected.  The
functions take and return torch tensors and never synchronise with the host.
"""

import math

import torch
from torch.utils._device import DeviceContext

from ... import _hip

__all__ = [
    "amax_layout", "kept_dims_first", "dense_flat_view", "absmax_accumulate", "reduce_amax_gpu", "fake_quant_int", "fake_quant_fp8",
    "ste_mask", "fake_quant_nvfp4", "fake_quant_block_fp", "mul_last_dim",
    "torch_is_intercepted",
]


def _prod(xs):
    return int(math.prod(xs))


def amax_layout(shape, keep_dims):
    """View a tensor of ``shape`` as [outer, axis, inner] such that the dims in ``keep_dims``
    (a contiguous run of dims, or none) form ``axis``.  Returns (outer, axis, inner) or None
    when the kept dims are not one contiguous run."""
    nd = len(shape)
    keep = sorted(d % nd for d in keep_dims if shape[d % nd] != 1)
    if not keep:
        return 1, 1, _prod(shape)
    if keep != list(range(keep[0], keep[-1] + 1)):
        # unit dims between kept dims do not break contiguity
        for d in range(keep[0], keep[-1] + 1):
            if d not in keep and shape[d] != 1:
                return None
    lo, hi = keep[0], keep[-1]
    return _prod(shape[:lo]), _prod(shape[lo:hi + 1]), _prod(shape[hi + 1:])


def kept_dims_first(x, keep_dims):
    """For kept dims that are not one contiguous run (2-D blocks: dims 0 and 2 of
    ``[N/b0, b0, K/b1, b1]``): a contiguous copy with the kept dims moved to the front, viewed by
    the kernels as [1, prod(kept), prod(rest)], and the permutation that was applied.  Costs one
    transposing copy each way; the common layouts never take this route."""
    nd = x.dim()
    keep = sorted({d % nd for d in keep_dims})
    perm = keep + [d for d in range(nd) if d not in keep]
    xp = x.permute(perm).contiguous()
    return xp, perm, (1, _prod(x.shape[d] for d in keep), _prod(xp.shape[len(keep):]))


def _undo_permutation(y, perm):
    inverse = [0] * len(perm)
    for i, d in enumerate(perm):
        inverse[d] = i
    return y.permute(inverse).contiguous()


def layout_from_amax_shape(x_shape, amax_shape):
    """[outer, axis, inner] for an amax whose shape broadcasts against ``x_shape`` (per-tensor,
    or equal to x on a contiguous run of dims and 1 elsewhere)."""
    n = _prod(amax_shape)
    if n == 1:
        return 1, 1, _prod(x_shape)
    a = list(amax_shape)
    if len(a) == 1 and len(x_shape) >= 1:
        # squeezed per-channel amax: the reference matches it to the dim of equal length
        if a[0] in list(x_shape):
            d = list(x_shape).index(a[0])
            return amax_layout(x_shape, [d])
        return None
    if len(a) != len(x_shape):
        return None
    keep = [d for d in range(len(a)) if a[d] != 1]
    if any(a[d] != x_shape[d] for d in keep):
        return None
    return amax_layout(x_shape, keep)


def dense_flat_view(x: torch.Tensor):
    """A 1-D view over the memory of ``x`` when ``x`` is a permutation of a contiguous block (a
    transposed K / V view, a channels-last tensor): every element appears exactly once, in memory
    order.  None when ``x`` has gaps or overlaps."""
    dims = sorted((d for d in range(x.dim()) if x.shape[d] != 1), key=lambda d: -x.stride(d))
    expect = 1
    for d in reversed(dims):
        if x.stride(d) != expect:
            return None
        expect *= x.shape[d]
    return x.as_strided((x.numel(),), (1,))


def absmax_accumulate(x: torch.Tensor, acc: torch.Tensor, layout, reread: bool = False):
    """acc (fp32, ``axis`` elements) = max(acc, abs-max of x over the reduced dims).  ``reread``:
    the caller reads ``x`` again right away (see ``_hip.absmax_into``)."""
    outer, axis, inner = layout
    if not x.is_contiguous():
        # a per-tensor maximum does not care about element order: a permuted dense tensor (the
        # [B, H, S, D] view of K / V) is reduced where it lies instead of through a copy
        flat = dense_flat_view(x) if axis == 1 else None
        x = flat if flat is not None else x.contiguous()
    return _hip.absmax_into(x, acc, outer, axis, inner, reread=reread)


def absmax_of(x: torch.Tensor, out_dtype: torch.dtype, reread: bool = False):
    """The abs-max of all of ``x`` as one element of ``out_dtype``; None where ``_hip.absmax_tensor`` does not
    apply (an accumulator and ``absmax_accumulate`` do)."""
    if not x.is_contiguous():
        flat = dense_flat_view(x)
        x = flat if flat is not None else x.contiguous()
    return _hip.absmax_tensor(x, out_dtype, reread=reread)


def reduce_amax_gpu(x: torch.Tensor, reduce_dims, keepdims=True, reread: bool = False):
    """``reduce_amax`` on the device: abs-max over ``reduce_dims`` (None = all) in x.dtype."""
    nd = x.dim()
    if reduce_dims is None:
        keep, out_shape = [], ()
    else:
        red = {d % nd for d in ([reduce_dims] if isinstance(reduce_dims, int) else reduce_dims)}
        keep = [d for d in range(nd) if d not in red]
        out_shape = tuple(1 if d in red else x.shape[d] for d in range(nd)) if keepdims else tuple(
            x.shape[d] for d in keep)
    layout = amax_layout(tuple(x.shape), keep)
    if layout is not None and layout[1] == 1 and x.is_cuda:
        whole = absmax_of(x, x.dtype, reread=reread)
        if whole is not None:
            return whole.reshape(out_shape)
    src = x
    if layout is None and x.is_cuda and x.is_contiguous():
        # one abs-max per two-dimensional block of a matrix: a workgroup per block, no transposed copy
        blocks = blocks2d_of(tuple(x.shape), keep)
        if blocks is not None and _hip.blocks2d_covered(x, *blocks):
            rows, cols, block_rows, block_cols = blocks
            acc = torch.zeros((rows // block_rows) * (cols // block_cols), dtype=torch.float32, device=x.device)
            _hip.absmax_blocks2d_into(x, acc, rows, cols, block_rows, block_cols)
            return acc.to(x.dtype).reshape(out_shape)
    if layout is None:
        src, _, layout = kept_dims_first(x, keep)
    acc = torch.zeros(layout[1], dtype=torch.float32, device=x.device)
    absmax_accumulate(src, acc, layout, reread=reread)
    return acc.to(x.dtype).reshape(out_shape)


def _qdq_layout(x, amax):
    return layout_from_amax_shape(tuple(x.shape), tuple(amax.shape))


def blocks2d_of(shape, kept) -> tuple | None:
    """``(rows, cols, block_rows, block_cols)`` when a contiguous tensor of ``shape`` whose scale
    dims are ``kept`` (a sorted list) is a matrix cut into two-dimensional blocks: the reshape
    ``[..., R, block_rows, C, block_cols]`` of ``[..., R * block_rows, C * block_cols]`` with a
    scale for every index of all dims but the two block dims (what a quantizer with block sizes
    on the last two dims sets up).  None otherwise."""
    nd = len(shape)
    if nd < 4 or list(kept) != [d for d in range(nd) if d not in (nd - 3, nd - 1)]:
        return None
    block_rows, block_cols = shape[nd - 3], shape[nd - 1]
    rows = math.prod(shape[:nd - 3]) * block_rows
    return rows, shape[nd - 2] * block_cols, block_rows, block_cols


def _qdq(x, amax, run, run2d=None):
    """``run(x2, amax_flat, outer, axis, inner)`` on ``x`` as it is when the amax spans one run
    of dims; ``run2d(x, amax_flat, rows, cols, block_rows, block_cols)`` when the amax is per
    two-dimensional block of a matrix; else ``run`` on a copy with the amax dims moved to the
    front (and moved back afterwards)."""
    x = x if x.is_contiguous() else x.contiguous()
    layout = _qdq_layout(x, amax)
    if layout is not None:
        return run(x, amax.reshape(-1).contiguous(), *layout)
    if amax.dim() != x.dim() or any(a not in (1, s) for a, s in zip(amax.shape, x.shape)):
        raise NotImplementedError(
            f"amax of shape {tuple(amax.shape)} does not broadcast against input {tuple(x.shape)}")
    if run2d is not None and x.is_cuda:
        blocks = blocks2d_of(tuple(x.shape), [d for d in range(x.dim()) if amax.shape[d] != 1])
        if blocks is not None and _hip.blocks2d_covered(x, *blocks):
            return run2d(x, amax.reshape(-1).contiguous(), *blocks)
    keep = [d for d in range(x.dim()) if amax.shape[d] != 1]
    xp, perm, layout = kept_dims_first(x, keep)
    y = run(xp, amax.reshape(-1).contiguous(), *layout)
    return _undo_permutation(y.view(xp.shape), perm)


with_scale_layout = _qdq   # the storage casts place their scales the same way


def fake_quant_int(x, amax, num_bits=8, unsigned=False, narrow_range=True):
    return _qdq(x, amax, lambda x2, a, outer, axis, inner: _hip.int_qdq(
        x2, a, outer, axis, inner, num_bits, unsigned, narrow_range),
        lambda x2, a, rows, cols, br, bc: _hip.int_qdq_blocks2d(
            x2, a, rows, cols, br, bc, num_bits, unsigned, narrow_range))


def fake_quant_fp8(x, amax=None, saturate=False):
    if amax is None:
        x = x if x.is_contiguous() else x.contiguous()
        return _hip.fp8_qdq(x, None, 1, 1, x.numel(), saturate)
    return _qdq(x, amax, lambda x2, a, outer, axis, inner: _hip.fp8_qdq(
        x2, a, outer, axis, inner, saturate),
        lambda x2, a, rows, cols, br, bc: _hip.fp8_qdq_blocks2d(x2, a, rows, cols, br, bc, saturate))


def ste_mask(x, amax, grad):
    """``torch.where(x.abs() <= amax, grad, 0)`` in one pass, or None where the kernel does not apply:
    mixed types, a gradient in another memory order, an amax on two separated runs of dims, a gradient
    that is itself differentiated (``create_graph``), batched or traced."""
    if (torch_is_intercepted() or (grad.requires_grad and torch.is_grad_enabled())
            or not torch._C._has_storage(grad)):
        return None
    if (type(grad) is not torch.Tensor or not (x.is_cuda and grad.is_cuda and amax.is_cuda) or x.dtype != grad.dtype or x.dim() == 0
            or x.shape != grad.shape or x.dtype not in _hip._DTYPES or amax.dtype not in _hip._DTYPES
            or not x.is_contiguous() or not grad.is_contiguous()):
        return None
    layout = (1, 1, x.numel()) if amax.numel() == 1 and amax.dim() <= x.dim() else None
    if layout is None and amax.dim() == x.dim():
        layout = _qdq_layout(x, amax)
    if layout is None:
        return None
    # a 0-dim amax takes the type of x in the comparison, one with dims promotes x to the wider type
    return _hip.ste_mask(x, grad, amax.reshape(-1).contiguous(), *layout,
                         narrow_amax=amax.dim() == 0 and amax.dtype != x.dtype)


def wgrad_mask_pays(tokens: int, n: int, k: int) -> bool:
    """Whether the weight gradient [n, k] over ``tokens`` is computed and masked in one pass.  The pass
    saved over the gradient outweighs the library's faster product up to 1024 tokens (one pass against two:
    14336 x 4096 bf16 165 us and 192, fp16 165 and 195; 4096 x 4096 57 and 57; at 2048 tokens 321 and 314), with
    fewer than 256 workgroups of 128 x 128 results up to 512 (512 x 512 10.7 us and 11.1, at 1024 tokens 17
    and 14; 16384 x 128 11.3 and 14.5, 18.5 and 17).  A tile that is mostly padding pays for less: 8 rows up to
    256 tokens (8 x 4096 fp16 6.8 us and 8.0, at 512 tokens 10.0 and 9.9), 8 or 16 columns, whose rows of the
    weight are 16 or 32 bytes, up to 64 (65536 x 8 bf16 7.6 us and 8.5, at 128 tokens 9.7 and 9.2; 24 columns 17
    and 21 at 512)."""
    most = 1024 if n * k >= 1 << 22 else 512
    if k < 24:
        most = 64
    elif n < 16:
        most = 256
    return 1 <= tokens <= most and n % 8 == 0 and k % 8 == 0


def input_grad_pays(tokens: int, n: int, k: int) -> bool:
    """Whether the input gradient of ``tokens`` rows behind a [n, k] weight is left to ``_hip.input_grad``.  us, it and the
    library's product, bf16 (fp16 is the same):

    up to 128 tokens k <= 32768 (14336 x 4096 at 128 tokens 34 and 125, 8192 x 28672 at 64 88 and 93, 4096 x 32768 at 100 51 and 55;
    wider results have tiles enough for the library: 4096 x 40960 at 64 78 and 70, 16384 x 53248 at 128 419 and 378);
    up to 256 tokens k <= 8192, or 16384 where n <= 16384 (16384 x 16384 at 192 tokens 135 and 184, 53248 x 8192 211 and 334; 8192 x 24576
    135 and 113, 28672 x 16384 at 192 233 and 226, 53248 x 14336 at 144 412 and 381);
    up to 512 tokens k <= 4096, or 6144 where n >= k, as a short sum does not pay for the partial sums (14336 x 4096 73 and 106, 6144 x 6144
    56 and 70; 4096 x 14336 66 and 62, 7168 x 7168 70 and 64);
    up to 1024 tokens k <= 4096 and n >= k (14336 x 4096 129 and 147, 4096 x 4096 45 and 46; 2752 x 4096 32 and 30, 5120 x 5120 85 and 76)."""
    if not 1 <= tokens <= 1024 or n % 8 or k % 8:
        return False
    if tokens <= 256:
        return k <= (32768 if tokens <= 128 else 16384 if n <= 16384 else 8192)
    return (k <= 4096 and (n >= k or tokens <= 512)) or (k <= 6144 and n >= k and tokens <= 512)


def fake_quant_nvfp4(x, global_amax, block_size=16, mode=0):
    x = x if x.is_contiguous() else x.contiguous()
    if global_amax.numel() != 1:
        global_amax = global_amax.amax()
    return _hip.nvfp4_qdq(x, global_amax.reshape(1), block_size, mode)


def fake_quant_block_fp(x, block_size, fmt, scale_fmt="E8M0", global_amax=None):
    """Block floating point fake quantisation along the last dim (``fused_amax_convert``):
    ``fmt`` / ``scale_fmt`` are format names (``"E4M3"``, ``"E2M1"``, ``"E8M0"`` ...)."""
    x = x if x.is_contiguous() else x.contiguous()
    if global_amax is not None:
        global_amax = global_amax.to(device=x.device, dtype=torch.float32).reshape(-1).contiguous()
    return _hip.block_fp_qdq(x, block_size, fmt, scale_fmt, global_amax)


def torch_is_intercepted() -> bool:
    """Whether something follows the tensor operations of this thread (a compiler, a dispatch or
    function mode, a functorch transform, forward-mode differentiation, a trace): a shortcut past an
    operator that it would see is not taken then.  The mode behind ``torch.set_default_device`` is no such
    thing: it is on the stack for a whole program and only says where new tensors go that name no device."""
    if torch.compiler.is_compiling():
        return True
    for i in range(torch._C._len_torch_function_stack()):
        if type(torch._C._get_function_stack_at(i)) is not DeviceContext:
            return True
    return bool(torch._C._len_torch_dispatch_stack() or torch._C._functorch.peek_interpreter_stack() is not None
                or torch.autograd.forward_ad._current_level >= 0 or torch._C._get_tracing_state() is not None)


def mul_last_dim(x, scale):
    """``x * scale`` for a scale that spans the last dim only."""
    x = x if x.is_contiguous() else x.contiguous()
    return _hip.mul_cols(x, scale.reshape(-1).contiguous())
