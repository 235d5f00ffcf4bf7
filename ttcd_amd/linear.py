"""Projections without a bias: y = x @ w.T, and the SwiGLU of a stacked gate|up
projection (host side of linear.hip).

Up to MAX_ROWS rows of x take the HIP kernels, everything else torch's GEMM
(hipBLASLt). Up to 64 rows the kernel is the faster on the GPU, up to 512 they
are about even (linear.hip has the times), and a call of it takes 7 us of host
time instead of 17, which is what a short prompt's layer is made of. Past 512
rows the GEMM runs longer than its call and is the faster of the two (4096 x
1024, 1000 rows: 17 / 13 us). Wide outputs (a vocabulary's logits) stay with
the GEMM, which streams them faster from 8 rows on (151936 x 1024: 78 / 61 us).
"""
from __future__ import annotations

import torch
import torch.autograd.forward_ad as fwAD
import torch.nn.functional as F

from . import _lib

_DT = {torch.bfloat16: _lib.DTYPE_BF16, torch.float16: _lib.DTYPE_F16}

MAX_ROWS = 512
MAX_COLS = 16384


def _rows_for_kernel(x: torch.Tensor, w: torch.Tensor) -> int:
    """The rows of x when the kernel takes x @ w.T, else 0."""
    if (type(x) is not torch.Tensor or type(w) not in (torch.Tensor, torch.nn.Parameter)
            or not x.is_cuda or x.device != w.device or x.dtype not in _DT or w.dtype != x.dtype
            or w.dim() != 2 or x.dim() < 1 or x.shape[-1] != w.shape[1] or w.shape[1] % 32
            or w.shape[0] > MAX_COLS or w.shape[0] < 1
            or (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad))
            or fwAD._current_level >= 0  # tangents are torch's to carry
            or not x.is_contiguous() or not w.is_contiguous()
            or x.data_ptr() % 16 or w.data_ptr() % 16):
        return 0
    rows = x.numel() // w.shape[1] if w.shape[1] else 0
    return rows if rows <= MAX_ROWS else 0


def _run(x: torch.Tensor, w: torch.Tensor, rows: int, cols: int, glu: int) -> torch.Tensor:
    K = w.shape[1]
    y = torch.empty(x.shape[:-1] + (cols,), dtype=x.dtype, device=x.device)
    _lib.check(_lib.lib().ttcd_linear_rows_fwd(x.data_ptr(), K, w.data_ptr(), y.data_ptr(), rows,
                                               cols, K, glu, _DT[x.dtype], _lib.stream(x)))
    return y


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """F.linear(x, w)."""
    rows = _rows_for_kernel(x, w)
    return _run(x, w, rows, w.shape[0], 0) if rows else F.linear(x, w)


def swiglu_linear(x: torch.Tensor, gate_up: torch.Tensor) -> torch.Tensor | None:
    """swiglu of the halves of F.linear(x, gate_up) in one launch, bit for bit the
    kernel's product and swiglu; None when the product is torch's."""
    rows = _rows_for_kernel(x, gate_up) if gate_up.shape[0] % 2 == 0 else 0
    return _run(x, gate_up, rows, gate_up.shape[0] // 2, 1) if rows else None
