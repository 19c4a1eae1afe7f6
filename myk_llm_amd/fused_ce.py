"""Fused linear + cross-entropy on MI355X (gfx950): the drop-in for myk-llm's
src/myk_llm/ops/fused_ce.py (exported by ops/__init__.py:2), same name, signature, defaults
and return values:

    fused_linear_cross_entropy(hidden, weight, targets, normalizer, z_loss=0.0,
                               ignore_index=-100, chunk_size=2048) -> (loss, ce_sum, z_sum)

loss = (sum of per-token CE + z_loss * sum of lse^2) / normalizer over supervised tokens;
ce_sum / z_sum are detached sums for logging (fused_ce.py:111-132). The (tokens, vocab)
logits are never materialized whole: tokens are processed in chunks, each chunk's logits
(hidden_chunk @ weight^T, bf16 GEMM with fp32 accumulation) are overwritten in place by the
gfx950 CE row kernel (csrc/fused_ce.hip, through the C ABI) with d loss / d logits, which the
next two GEMMs fold into the hidden and weight gradients at once. As in the reference the
gradient is computed during the forward pass, so the loss is backpropagated exactly once.

The products are libmykfa.so's (csrc/gemm.hip) where the hidden size is a multiple of 8, else
torch.matmul's. The weight gradient accumulates in fp32 inside its product instead of rounding each
chunk's bf16 product before an fp32 add (fused_ce.py:89). Without a chunk_size a pass there holds as many
tokens as _KEEP_BYTES of d logits do (the default's 2048 where the device's memory holds no more).
"""

from __future__ import annotations

import ctypes
import operator
from typing import cast

import torch
from torch import Tensor
from torch.autograd import forward_ad

from . import _lib
from .flash_attn import _DeviceGuard, _dtype_code, _same_device, _stream
from .gemm import gemm, usable


def _ce_rows(logits: Tensor, targets: Tensor, ce: Tensor, lse: Tensor, scale: float, z_coef: float,
             ignore_index: int) -> None:
    """The row kernel on one chunk: lse, ce, and logits := d loss / d logits, in place."""
    p = _lib.CeParams()
    p.logits, p.targets, p.ce, p.lse = logits.data_ptr(), targets.data_ptr(), ce.data_ptr(), lse.data_ptr()
    p.row_stride, p.rows, p.vocab = logits.stride(0), logits.shape[0], logits.shape[1]
    p.ignore_index = int(ignore_index)
    p.scale, p.z_coef = float(scale), float(z_coef)
    p.dtype = _dtype_code(logits.dtype)
    _lib.check(_lib.lib().mykfa_ce_rows(ctypes.byref(p), _stream(logits.device)))


def _accumulate_fp32(acc: Tensor, a: Tensor, b: Tensor) -> None:
    """acc (fp32) += a @ b with bf16 operands, accumulated in fp32 by the GEMM itself."""
    torch.ops.aten.addmm.dtype_out(acc, a, b, torch.float32, beta=1, alpha=1, out=acc)


def _chunk_spans(n: int, size: int) -> list[tuple[int, int]]:
    return [(lo, min(lo + size, n)) for lo in range(0, n, size)]


# d logits in memory at once. One pass's products run over all its tokens: fewer rounds of workgroups
# cut short, fewer fp32 partials of d hidden, and the fp32 d weight is read and written once per pass
# (65536 x 1024 over 8192 tokens 990 us at once, 4 x 335 in chunks of 2048). Whole head, chunks of 2048
# with up to 1 GiB kept for d weight alone, against passes of up to this: 16384 tokens of hidden 1024 and
# vocabulary 65536 7280 -> 7000 us (1.5 GiB the same, 1 GiB 7370: three passes), 32000 3510 -> 3365; 512 and 8000
# 836 -> 638; 3000 tokens of 1024 and 32000 750 -> 725.
_KEEP_BYTES = 5 << 28


class _Unset(int):
    """chunk_size's default: its value in a signature, and not a caller's wish."""


_CHUNK = _Unset(2048)


def _pass_rows(tokens: int, row_bytes: int, chunk_size: int) -> int:
    """Tokens per pass: chunk_size where the caller gave one, which bounds the memory of its d logits. Else
    even passes over all of them, whole 256-row tiles where that fits, of at most _KEEP_BYTES of d logits or
    the default's tokens, whichever is more."""
    if not isinstance(chunk_size, _Unset):
        return min(operator.index(chunk_size), tokens)
    most = max(chunk_size, _KEEP_BYTES // row_bytes)
    passes = -(-tokens // most)
    return min(tokens, most, (-(-tokens // passes) + 255) // 256 * 256)


def _operand(x: Tensor) -> Tensor:
    """x in bf16 rows that the products read, at most 2^22 elements apart (a tile's 256 within 2 GiB). A clone
    and not contiguous(), which hands back a contiguous tensor that starts off 16 bytes, or a single row of
    an odd stride, as it is."""
    if x.dtype != torch.bfloat16:
        x = x.to(torch.bfloat16)
    return x if usable(x) and x.stride(0) <= 1 << 22 else x.clone(memory_format=torch.contiguous_format)


def _loss_and_gradients(hidden: Tensor, weight: Tensor, targets: Tensor, scale: float, z_coef: float,
                        ignore_index: int, chunk_size: int) -> tuple[Tensor, Tensor, Tensor]:
    """One pass over the tokens in chunks. Returns (row_stats, d_hidden, d_weight):
    row_stats[0] / row_stats[1] are every token's cross-entropy and natural-log LSE (fp32),
    d_hidden (bf16) and d_weight (fp32) the gradients of the loss for an upstream gradient of 1.

    Per chunk: the logits product writes a (rows, vocab) bf16 block, the gfx950 row kernel turns
    that block into d loss / d logits in place while producing the row statistics, and the
    same block then feeds the two gradient products. d_weight is accumulated in fp32 by the
    product (beta = 1) so no partial sum is ever rounded to bf16."""
    dev = hidden.device
    tokens, width = hidden.shape
    vocab = weight.shape[0]
    w16 = weight if weight.dtype == torch.bfloat16 else weight.to(torch.bfloat16)
    row_stats = torch.empty((2, tokens), dtype=torch.float32, device=dev)
    d_hidden = torch.empty((tokens, width), dtype=torch.bfloat16, device=dev)
    tgt = targets if targets.dtype == torch.int64 else targets.to(torch.int64)
    # Rows of the d logits start a 128-byte line each, an odd multiple of 256 bytes apart: rows a power
    # of two apart fall on few channels (2048 x 65536 x 1024 in / out: logits 291 -> 268 us, d hidden
    # 265 -> 251; rows off the lines 325 and 276).
    stride = ((vocab + 127) // 128 | 1) * 128
    # (A weight of another width is left to torch.mm, which refuses it: mykfa_gemm takes the sizes it is told.)
    if (width % 8 == 0 and width > 0 and vocab > 0 and tokens > 0 and max(stride, width) < 1 << 22
            and tuple(weight.shape) == (vocab, width)):
        w16 = _operand(w16)
        d_weight = torch.empty((vocab, width), dtype=torch.float32, device=dev)
        chunk = min(chunk_size, tokens)
        rows = _pass_rows(tokens, 2 * stride, chunk_size)

        def run(rows: int) -> None:
            blocks = torch.empty((rows, stride), dtype=torch.bfloat16, device=dev)
            for lo, hi in _chunk_spans(tokens, rows):
                block, h = blocks[:hi - lo, :vocab], _operand(hidden[lo:hi])
                gemm(h, w16, block, hi - lo, vocab, width, b_transposed=True)
                _ce_rows(block, tgt[lo:hi], row_stats[0, lo:hi], row_stats[1, lo:hi], scale, z_coef, ignore_index)
                gemm(block, w16, d_hidden[lo:hi], hi - lo, width, vocab)
                gemm(block, h, d_weight, vocab, width, hi - lo, a_transposed=True, beta=0.0 if lo == 0 else 1.0)

        try:
            run(rows)
        except torch.OutOfMemoryError:
            if rows <= chunk:
                raise
            rows = 0
        if rows == 0:  # past the handler, which holds the larger buffer
            run(chunk)
        return row_stats, d_hidden, d_weight
    d_weight = torch.zeros(weight.shape, dtype=torch.float32, device=dev)
    for lo, hi in _chunk_spans(tokens, chunk_size):
        h16 = hidden[lo:hi]
        if h16.dtype != torch.bfloat16:
            h16 = h16.to(torch.bfloat16)
        block = torch.mm(h16, w16.t())
        _ce_rows(block, tgt[lo:hi], row_stats[0, lo:hi], row_stats[1, lo:hi], scale, z_coef, ignore_index)
        torch.mm(block, w16, out=d_hidden[lo:hi])
        _accumulate_fp32(d_weight, block.t(), h16)
    return row_stats, d_hidden, d_weight


_SCALE_DTYPES = {torch.bfloat16: _lib.DTYPE_BF16, torch.float16: _lib.DTYPE_FP16, torch.float32: _lib.DTYPE_FP32}


def _loss_of(row_stats: Tensor, scale: float, z_coef: float) -> tuple[Tensor, Tensor, Tensor]:
    """(loss, ce_sum, z_sum) of the tokens' statistics."""
    if row_stats.shape[1] > 1 << 17:  # more than one workgroup should sum
        ce_sum = row_stats[0].sum()
        z_sum = torch.dot(row_stats[1], row_stats[1])
        return torch.add(ce_sum, z_sum, alpha=z_coef) * scale, ce_sum, z_sum
    out = tuple(row_stats.new_empty(()) for _ in range(3))
    ce = row_stats.data_ptr()
    p = _lib.CeLossParams(ce, ce + 4 * row_stats.shape[1], *(x.data_ptr() for x in out), row_stats.shape[1], scale, z_coef)
    with _DeviceGuard(row_stats.device):
        _lib.check(_lib.lib().mykfa_ce_loss(ctypes.byref(p), _stream(row_stats.device)))
    return out


def _plain(x: Tensor) -> bool:
    """Whether x's values are the memory behind it: no subclass, mapped or wrapped tensor, no tangent."""
    return (type(x) is Tensor and not torch._C._functorch.is_functorch_wrapped_tensor(x)
            and not torch._C._functorch.is_legacy_batchedtensor(x)
            and (forward_ad._current_level < 0 or forward_ad.unpack_dual(x).tangent is None))


def _scaled(grad: Tensor, upstream: Tensor, dtype: torch.dtype) -> Tensor:
    """grad * upstream, rounded to grad's type, as dtype. The kernel takes the gradients as the forward left
    them; what a hook on saved tensors made of them, a gradient of the gradient, or a mapped or dual one goes
    through torch."""
    if (grad.dtype not in (torch.bfloat16, torch.float32) or dtype not in _SCALE_DTYPES or upstream.dtype != torch.float32
            or upstream.device != grad.device or torch.is_grad_enabled() or not _plain(grad) or not _plain(upstream)
            or not grad.is_contiguous() or grad.data_ptr() % 16 or upstream.numel() != 1):
        return grad.mul(upstream).to(dtype)
    out = torch.empty_like(grad, dtype=dtype)
    p = _lib.ScaleParams(grad.data_ptr(), out.data_ptr(), upstream.data_ptr(), grad.numel(), _SCALE_DTYPES[grad.dtype],
                         _SCALE_DTYPES[dtype])
    with _DeviceGuard(grad.device):
        _lib.check(_lib.lib().mykfa_scale(ctypes.byref(p), _stream(grad.device)))
    return out


class _LinearCrossEntropy(torch.autograd.Function):
    """The loss and both gradients come out of the forward (the reference's scheme,
    fused_ce.py:70-108): the backward only multiplies the stored gradients by the upstream
    gradient of the loss and casts them to the parameters' dtypes."""

    @staticmethod
    def forward(ctx, hidden, weight, targets, normalizer, z_coef, ignore_index, chunk_size):  # pyright: ignore[reportIncompatibleMethodOverride]
        scale = 1.0 / normalizer
        with torch.autocast(device_type="cuda", enabled=False), _DeviceGuard(hidden.device):
            row_stats, d_hidden, d_weight = _loss_and_gradients(hidden, weight, targets, scale, z_coef,
                                                                ignore_index, chunk_size)
        loss, ce_sum, z_sum = _loss_of(row_stats, scale, z_coef)
        ctx.save_for_backward(d_hidden, d_weight)
        ctx.grad_dtypes = (hidden.dtype, weight.dtype)
        ctx.mark_non_differentiable(ce_sum, z_sum)
        return loss, ce_sum, z_sum

    @staticmethod
    def backward(ctx, upstream, _unused_ce, _unused_z):  # pyright: ignore[reportIncompatibleMethodOverride]
        d_hidden, d_weight = ctx.saved_tensors
        hidden_dtype, weight_dtype = ctx.grad_dtypes
        return (_scaled(d_hidden, upstream, hidden_dtype), _scaled(d_weight, upstream, weight_dtype),
                None, None, None, None, None)


def fused_linear_cross_entropy(hidden: Tensor, weight: Tensor, targets: Tensor, normalizer: float,
                               z_loss: float = 0.0, ignore_index: int = -100,
                               chunk_size: int = _CHUNK) -> tuple[Tensor, Tensor, Tensor]:
    """Returns (loss, ce_sum, z_sum): loss = (sum CE + z_loss * sum lse^2) / normalizer
    (fused_ce.py:111-132). hidden (..., H), weight (V, H), targets (...) integer class ids
    with ignore_index marking unsupervised tokens. A chunk_size is the most tokens whose d logits are in
    memory at once; without one up to 1.25 GiB of them are, where the device has that."""
    if not hidden.is_cuda:
        raise RuntimeError("fused cross entropy is CUDA-only")
    _same_device(hidden.device, weight=weight, targets=targets)
    if chunk_size <= 0:
        raise ValueError(f"chunk_size must be positive; got {chunk_size}")
    result = _LinearCrossEntropy.apply(hidden.reshape(-1, hidden.size(-1)), weight, targets.reshape(-1),
                                       float(normalizer), float(z_loss), ignore_index, chunk_size)
    return cast(tuple[Tensor, Tensor, Tensor], result)
