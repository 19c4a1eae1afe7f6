"""Matrix products through libmykfa.so (csrc/gemm.hip): what fused_ce.py and muon.py multiply with.
bf16 operands, fp32 accumulation; operands and results as (rows, cols) or (batch, rows, cols)
tensors whose layout satisfies mykfa_gemm (include/mykfa.h)."""

from __future__ import annotations

import ctypes
from typing import Optional

import torch
from torch import Tensor

from . import _lib
from .flash_attn import _stream


def usable(x: Tensor) -> bool:
    """Rows that mykfa_gemm can read: contiguous last dimension, 16-byte aligned, strides
    multiples of 8, each row at least its columns rounded up to 8 elements long."""
    s = x.stride()
    return (s[-1] == 1 and x.data_ptr() % 16 == 0 and all(v % 8 == 0 for v in s[:-1])
            and s[-2] >= (x.shape[-1] + 7) // 8 * 8)


def _layout(x: Optional[Tensor]) -> tuple[int, int]:
    if x is None:
        return 0, 0
    s = x.stride()
    return (0, s[0]) if len(s) == 2 else (s[0], s[1])


def gemm(a: Tensor, b: Optional[Tensor], c: Tensor, m: int, n: int, k: int, *, a_transposed: bool = False,
         b_transposed: bool = False, symmetric: bool = False, add: Optional[Tensor] = None, alpha: float = 1.0,
         beta: float = 0.0) -> None:
    """c = alpha * op(a) op(b) + beta * add (bf16 c), or c = op(a) op(b) + beta * c (fp32 c), on
    torch's current stream of the current device. symmetric: b = a^T."""
    buf = bytearray(_lib.GEMM_PACK.size)
    _lib.GEMM_PACK.pack_into(
        buf, 0, a.data_ptr(), 0 if b is None else b.data_ptr(), 0 if add is None else add.data_ptr(), c.data_ptr(),
        *_layout(a), *_layout(b), *_layout(add), *_layout(c), a.shape[0] if a.dim() == 3 else 1, m, n, k,
        a_transposed, b_transposed, symmetric, alpha, beta,
        _lib.DTYPE_FP32 if c.dtype == torch.float32 else _lib.DTYPE_BF16)
    p = _lib.GemmParams.from_buffer(buf)
    L = _lib.lib()
    nbytes = L.mykfa_gemm_workspace_size(ctypes.byref(p))
    ws = torch.empty(nbytes, dtype=torch.uint8, device=a.device) if nbytes else None
    _lib.check(L.mykfa_gemm(ctypes.byref(p), None if ws is None else ws.data_ptr(), nbytes, _stream(a.device)))
