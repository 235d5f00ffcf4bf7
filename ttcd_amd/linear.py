"""Projections without a bias: y = x @ w.T, and the SwiGLU of a stacked gate|up
projection (host side of linear.hip).

`linear` and `swiglu_linear` run the HIP kernels wherever these take the call
(up to MAX_ROWS rows of x). `project` and `swiglu_project`, which the layers
call, run them where they are also the faster on the GPU (`_pays`), and else
torch's GEMM (hipBLASLt). Wide outputs (a vocabulary's logits) stay with the
GEMM, which streams them faster from 8 rows on (151936 x 1024: 78 / 61 us).
"""
from __future__ import annotations

import torch
import torch.autograd.forward_ad as fwAD
import torch.nn.functional as F

from . import _lib

_DT = {torch.bfloat16: _lib.DTYPE_BF16, torch.float16: _lib.DTYPE_F16}

_WEIGHTS = (torch.Tensor, torch.nn.Parameter)

MAX_ROWS = 512
MAX_COLS = 16384


def _rows_for_kernel(x: torch.Tensor, w: torch.Tensor) -> int:
    """The rows of x when the kernel takes x @ w.T, else 0."""
    if type(x) is not torch.Tensor or type(w) not in _WEIGHTS:
        return 0
    xs, ws, n = x.shape, w.shape, x.numel()
    if len(ws) != 2 or not xs or n > MAX_ROWS * ws[1]:
        return 0  # a long call pays for no more than this
    N, K = ws
    dtype = x.dtype
    if (xs[-1] != K or K % 32 or K < 1 or N > MAX_COLS or N < 1
            or dtype not in _DT or w.dtype != dtype or not x.is_cuda or x.device != w.device
            or (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad))
            or fwAD._current_level >= 0  # tangents are torch's to carry
            # and so are autocast's casts
            or (torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") != dtype)
            or not x.is_contiguous() or not w.is_contiguous()
            or x.data_ptr() % 16 or w.data_ptr() % 16):
        return 0
    return n // K


def _run(x: torch.Tensor, w: torch.Tensor, rows: int, cols: int, glu: int) -> torch.Tensor:
    K = w.shape[1]
    y = torch.empty(x.shape[:-1] + (cols,), dtype=x.dtype, device=x.device)
    _lib.check(_lib.lib().ttcd_linear_rows_fwd(x.data_ptr(), K, w.data_ptr(), y.data_ptr(), rows,
                                               cols, K, glu, _DT[x.dtype], _lib.stream(x)))
    return y


def _pays(M: int, N: int, K: int, glu: bool) -> bool:
    """Whether the kernel's time on the GPU is about that of the GEMM (and of the
    swiglu launch after it, if glu) or less, for M rows of x and w (N, K).

    GPU time alone, so that a call in a captured graph or behind queued work is
    not the slower one; a short prompt's call has 8 us of host time by the
    kernel (3.6 of them in the C entry) and 19 by the GEMM on top. Measured
    kernel / GEMM over N = 256..16384 and K = 96..11008, weights not in a cache
    (us):
    * up to 16 rows W is read once: faster up to 4096 columns at any K (4096 x
      11008, 16 rows, 32 / 39) and up to 2^23 weights beyond (6144 x 1024 6.7 / 8.2;
      6144 x 3072 1.3 times, 16384 x 4096 45 / 33);
    * up to 64 rows every 16 columns read x again, and the time grows with
      columns times rows: 4096 x 1024, 64 rows, 7.8 / 11.7 and 1024 x 3072 8.5 / 12,
      but 6144 x 1024 12.5 / 11.9 and 4096 x 4096 25 / 15. The SwiGLU form has half
      the columns per weight: 6144 x 1024, 64 rows, 11.5 / 14.5;
    * past 64 rows a 64 x 64 tile's chain over K is the call until tiles outnumber
      the CUs: 4096 x 1024, 512 rows, 11.2 / 13.1, but 8192 x 1024, 384 rows,
      1.2 times. A long K over few tiles leaves most CUs idle where the GEMM
      splits K: 1024 x 3072, 128 rows, 16.4 / 9.8, but 300 rows 15.2 / 15.3; the
      worst that is left to the kernel, 1024 x 2048, 65 to 256 rows, 9.5 / 8.3.
      K that is no multiple of 64 has no tiles: 4096 x 1056, 256 rows, 20 / 14.
    Of 292 calls drawn from these ranges that go to the kernel the median took 0.69
    of the GEMM's time and six more than 1.1 (1.4 at most, 28 rows, 2060 x 3072).
    """
    if K > 4096 and K > 4 * N:
        return False  # 384 x 6016, 2 rows: 18.7 / 13.9
    if M <= 16:
        return N <= 4096 or N * K <= 1 << 23
    if M <= 64:
        reads = -(-M // 16) * N
        room = 1.5 if glu and K <= 1024 else 1
        return N <= 1024 or (reads <= room * (1 << 14) and reads * K <= room * (1 << 24))
    if K % 64:
        return False
    tiles = -(-N // 64) * -(-M // 64)
    if K <= 1024:
        return tiles <= (1536 if glu else 576)
    if glu:
        return N >= 3072 and K <= 2048 and tiles <= 1024
    return tiles <= 256 and (K <= 2048 or N >= K or (K <= 3072 and tiles >= 80))


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """F.linear(x, w), by the kernel where it takes the call."""
    rows = _rows_for_kernel(x, w)
    return _run(x, w, rows, w.shape[0], 0) if rows else F.linear(x, w)


def swiglu_linear(x: torch.Tensor, gate_up: torch.Tensor) -> torch.Tensor | None:
    """swiglu of the halves of F.linear(x, gate_up) in one launch, bit for bit the
    kernel's product and swiglu; None when the kernel does not take the call."""
    rows = _rows_for_kernel(x, gate_up) if gate_up.shape[0] % 2 == 0 else 0
    return _run(x, gate_up, rows, gate_up.shape[0] // 2, 1) if rows else None


def project(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """F.linear(x, w), by the faster of the kernel and the GEMM."""
    rows = _rows_for_kernel(x, w)
    if rows and _pays(rows, w.shape[0], w.shape[1], False):
        return _run(x, w, rows, w.shape[0], 0)
    return F.linear(x, w)


def swiglu_project(x: torch.Tensor, gate_up: torch.Tensor) -> torch.Tensor | None:
    """swiglu_linear where it is faster than the GEMM and a swiglu launch, else None:
    also for the widths that swiglu refuses (no multiple of 8), whatever the rows."""
    rows = _rows_for_kernel(x, gate_up) if gate_up.shape[0] % 16 == 0 else 0
    if rows and _pays(rows, gate_up.shape[0], gate_up.shape[1], True):
        return _run(x, gate_up, rows, gate_up.shape[0] // 2, 1)
    return None
