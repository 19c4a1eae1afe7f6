"""Muon's batched Gram products on MI355X (gfx950): the drop-in for the batched SYRK of
myk-llm's src/myk_llm/ops/muon.py (exported by ops/__init__.py), same names and arguments:

    batched_syrk(x, bias=None, alpha=1.0, beta=0.0, out=None) -> out
        out[b] = alpha * x[b] @ x[b]^T + beta * bias[b] in bf16, computing only the
        lower-triangular tiles and mirroring them (ops/muon.py:28-143)
    batched_newton_schulz_orthogonalize(packed, steps, transposed=None, norm_sq=None, eps=1e-7)
        the quintic Newton-Schulz iteration on a batch of matrices (ops/muon.py:218-268):
        per step G = X X^T and G2 = b G + c G G through batched_syrk, X' = a X + G2 X

Every product runs in the hand-written gfx950 kernels of libmykfa.so (csrc/gemm.hip); the whole
iteration is one call of its C ABI (csrc/muon.hip: norms, scaled copy, three products a step).

Differences from the reference's layout handling: the kernel reads k-contiguous rows whose
length is a multiple of 8, so transposed or strided x and unaligned k are copied once
(zero-padded) before the call; the Newton-Schulz driver iterates tall matrices on a transposed
copy instead of transposed views.
"""

from __future__ import annotations

import ctypes
from typing import Optional

import torch
from torch import Tensor

from . import _lib
from .flash_attn import _DeviceGuard, _same_device, _stream
from .gemm import gemm, usable

NS_COEFFICIENTS = (3.4445, -4.7750, 2.0315)  # ops/muon.py:25


def _kernel_x(x: Tensor) -> Tensor:
    """x as (B, M, Kp) bf16 rows with Kp a multiple of 8, 16-byte aligned, row stride 8k."""
    b, m, k = x.shape
    kp = (k + 7) // 8 * 8
    if kp == k and usable(x):
        return x
    xp = torch.zeros((b, m, kp), dtype=torch.bfloat16, device=x.device)
    xp[..., :k] = x
    return xp


def batched_syrk(x: Tensor, bias: Optional[Tensor] = None, alpha: float = 1.0, beta: float = 0.0,
                 out: Optional[Tensor] = None) -> Tensor:
    """alpha * (x @ x.transpose(-2, -1)) + beta * bias for bf16 x of shape (B, M, K)
    (ops/muon.py:107-143). Only the lower-triangular tiles are evaluated and mirrored, so a
    given bias is assumed symmetric (as in the reference)."""
    if not x.is_cuda:
        raise RuntimeError("batched SYRK is CUDA-only: x must be a GPU (HIP) tensor")
    if x.dtype != torch.bfloat16:
        raise TypeError(f"batched SYRK needs bf16 x; got {x.dtype}")
    if x.dim() != 3:
        raise ValueError(f"x must be (batch, m, k); got {tuple(x.shape)}")
    B, M, _ = x.shape
    _same_device(x.device, bias=bias, out=out)
    if out is None:
        out = torch.empty((B, M, M), device=x.device, dtype=torch.bfloat16)
    if out.shape != (B, M, M) or out.dtype != torch.bfloat16:
        raise ValueError(f"out must be bf16 ({B}, {M}, {M}); got {out.dtype} {tuple(out.shape)}")
    if bias is not None and (bias.shape != (B, M, M) or bias.dtype != torch.bfloat16):
        raise ValueError(f"bias must be bf16 ({B}, {M}, {M}); got {bias.dtype} {tuple(bias.shape)}")
    xk = _kernel_x(x)
    o = out
    if not (o.stride(2) == 1 and o.stride(1) % 4 == 0 and o.data_ptr() % 8 == 0 and o.stride(1) >= M):
        # the kernel's mirrored stores are 8 bytes wide: rows padded to a multiple of 4
        o = torch.empty((B, M, (M + 3) // 4 * 4), device=x.device, dtype=torch.bfloat16)[:, :, :M]
    if bias is not None and (bias.stride(2) != 1 or bias.data_ptr() % 2):
        bias = bias.contiguous()
    if B > 0 and M > 0:
        with _DeviceGuard(x.device):
            gemm(xk, None, o, M, M, xk.shape[2], symmetric=True, add=bias, alpha=float(alpha), beta=float(beta))
    if o is not out:
        out.copy_(o)
    return out


def _frobenius_norm(packed: Tensor) -> Tensor:
    """Per-matrix Frobenius norm in fp32 of contiguous (B, rows, cols), as
    torch.linalg.vector_norm(packed, dim=(-2, -1), dtype=torch.float32) (ops/muon.py:241) but
    reduced in two levels (256 partial norms per matrix, then their root sum of squares): a
    single reduction with only B outputs runs on a handful of workgroups on this platform
    (measured 688 us for 9 x 1024 x 4096 bf16)."""
    B = packed.shape[0]
    flat = packed.view(B, -1)
    parts = 256 if flat.shape[1] % 256 == 0 and flat.shape[1] >= 256 * 1024 else 1
    partial = torch.linalg.vector_norm(flat.view(B, parts, -1), dim=-1, dtype=torch.float32)
    return partial.square().sum(-1).sqrt() if parts > 1 else partial[:, 0]


def batched_newton_schulz_orthogonalize(packed: Tensor, steps: int, transposed: Optional[bool] = None,
                                        norm_sq: Optional[Tensor] = None, eps: float = 1e-7) -> Tensor:
    """Batched quintic Newton-Schulz on packed (B, rows, cols) in bf16 (ops/muon.py:218-268).

    With norm_sq (per-matrix squared Frobenius norm of packed) the input is scaled by
    1 / max(sqrt(norm_sq), eps) in place, as the reference's _scale_bf16_kernel does;
    otherwise its norm is computed first. Returns a contiguous (B, rows, cols) tensor."""
    a, b, c = NS_COEFFICIENTS
    if packed.dtype != torch.bfloat16:
        packed = packed.bfloat16()
    if not packed.is_contiguous():
        packed = packed.contiguous()
    B, rows, cols = packed.shape
    if transposed is None:
        transposed = rows > cols
    if norm_sq is not None:
        inv = 1.0 / torch.clamp(norm_sq.reshape(B, 1, 1).float().sqrt(), min=eps)
        packed.copy_((packed.float() * inv).bfloat16())
    if steps <= 0 or packed.numel() == 0:
        if norm_sq is None:
            packed = (packed / _frobenius_norm(packed).reshape(B, 1, 1).clamp_(min=eps)).bfloat16()
        return packed
    if not packed.is_cuda:
        raise RuntimeError("batched Newton-Schulz is CUDA-only: packed must be a GPU (HIP) tensor")
    if torch.is_grad_enabled() and packed.requires_grad:
        raise RuntimeError("batched Newton-Schulz has no gradient: packed must not require one")
    out = torch.empty_like(packed)
    p = _lib.NewtonSchulzParams(packed.data_ptr(), out.data_ptr(), B, rows, cols, bool(transposed),
                                norm_sq is not None, steps, a, b, c, eps)
    L = _lib.lib()
    with _DeviceGuard(packed.device):
        ws = torch.empty(L.mykfa_newton_schulz_workspace_size(ctypes.byref(p)), dtype=torch.uint8, device=packed.device)
        _lib.check(L.mykfa_newton_schulz(ctypes.byref(p), ws.data_ptr(), ws.numel(), _stream(packed.device)))
    return out
