"""Projections of few rows (ttcd_amd.linear): the kernel against 64 bits at the
edges of its tiles, its SwiGLU form against its own product, and what is left
to torch.

Bound: the fp32 sum of K products is off by at most K 2^-24 of the sum of their
magnitudes, and the result is rounded once, u |y|."""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from ttcd_amd import _lib, linear as L, ttt


def _xw(shape, N, K, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(*shape, K, generator=g).to(dtype).cuda()
    return x, (torch.randn(N, K, generator=g) * K ** -0.5).to(dtype).cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("shape,N,K,dtype", [
    ((1,), 16, 32, torch.bfloat16), ((1, 16), 24, 96, torch.float16), ((2, 8), 1, 1024, torch.bfloat16),
    ((17,), 1000, 960, torch.bfloat16), ((3, 11), 4096, 1024, torch.bfloat16),
    ((1, 64), 1024, 3072, torch.float16), ((48,), 8200, 256, torch.bfloat16),
    ((64,), 6144, 1056, torch.bfloat16), ((40,), 8192, 128, torch.bfloat16),
    # 64 x 64 tiles: one step, an odd number of steps for two groups, both sides
    # of 256 tiles, ragged rows and columns; K that tiles do not take
    ((65,), 64, 64, torch.bfloat16), ((2, 50), 1000, 576, torch.float16), ((129,), 66, 448, torch.bfloat16),
    ((512,), 1024, 3072, torch.bfloat16), ((3, 100), 6144, 1024, torch.bfloat16),
    ((65,), 16384, 960, torch.float16), ((511,), 3, 512, torch.bfloat16), ((70,), 96, 96, torch.bfloat16)])
@torch.inference_mode()
def test_few_rows_match_64_bits(gpu, shape, N, K, dtype):
    x, w = _xw(shape, N, K, dtype, N + K)
    got = L.linear(x, w)
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    want = x.double() @ w.double().T
    limit = u * want.abs() + K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert got.shape == shape + (N,) and got.dtype == dtype
    assert ((got.double() - want).abs() <= limit).all()
    if N % 2 == 0 and N % 16 == 0:
        z = L.swiglu_linear(x, w)
        assert torch.equal(z, ttt.swiglu(got[..., :N // 2], got[..., N // 2:]))


@pytest.mark.gpu
def test_what_is_left_to_torch(gpu):
    x, w = _xw((513,), 64, 64, torch.bfloat16, 1)
    assert L._rows_for_kernel(x[:512], w) == 512
    for a, b in ((x, w), (x[:8, :48], w[:, :48]), (x[:8].float(), w.float()), (x[:64].t(), w),
                 (x[:8], w[::2]), (x.flatten()[1:65].view(1, 64), w), (x[:0], w)):
        assert L._rows_for_kernel(a, b) == 0
        assert torch.equal(L.linear(a, b), F.linear(a, b))
        assert L.swiglu_linear(a, b) is None
    wg = w.clone().requires_grad_()
    y = L.linear(x[:8], wg)
    assert y.requires_grad and L._rows_for_kernel(x[:8], wg) == 0
    with torch.no_grad():
        assert L._rows_for_kernel(x[:8], wg) == 8
    with torch.autograd.forward_ad.dual_level():
        assert L._rows_for_kernel(x[:8], w) == 0


def test_cpu_tensors_and_bad_arguments():
    x, w = torch.randn(4, 64), torch.randn(8, 64)
    assert torch.equal(L.linear(x, w), F.linear(x, w))
    C, P = _lib.lib(), 0x10000
    call = lambda x=P, st=64, w=P, M=4, N=8, K=64, dt=0: C.ttcd_linear_rows_fwd(  # noqa: E731
        x, st, w, P, M, N, K, 0, dt, None)
    assert call(x=None) == call(M=0) == call(st=32) == _lib.TTCD_ERR_INVALID_ARGUMENT
    assert call(K=48) == call(dt=2) == call(w=P + 2) == call(st=65) == _lib.TTCD_ERR_UNSUPPORTED


def test_the_kernel_is_chosen_by_shape():
    """Both sides of the lines that the kernel's and the GEMM's times draw (_pays)."""
    kernel = [(1, 4096, 11008, 0), (16, 6144, 1024, 0), (64, 1024, 3072, 0), (64, 4096, 1024, 0),
              (64, 6144, 1024, 1), (65, 1024, 2048, 0), (512, 4096, 1024, 0), (384, 6144, 1024, 0),
              (512, 6144, 1024, 1), (256, 4096, 4096, 0), (300, 1024, 3072, 0)]
    gemm = [(16, 16384, 4096, 0), (17, 4096, 11008, 0), (64, 6144, 1024, 0), (64, 4096, 4096, 0),
            (65, 1024, 3072, 0), (256, 1024, 3072, 0), (128, 960, 2560, 0), (2, 384, 6016, 1),
            (512, 6144, 1024, 0), (512, 8192, 1024, 0), (300, 4096, 4096, 0), (128, 2048, 2048, 1), (256, 4096, 1056, 0)]
    assert [c for c in kernel if not L._pays(*c)] == [] and [c for c in gemm if L._pays(*c)] == []


@pytest.mark.gpu
@torch.inference_mode()
def test_project_is_the_kernel_or_torch(gpu):
    for M, N, K, pays in ((128, 4096, 1024, True), (128, 1024, 3072, False)):
        x, w = _xw((M,), N, K, torch.bfloat16, M)
        assert torch.equal(L.project(x, w), L.linear(x, w) if pays else F.linear(x, w))
        z = L.swiglu_project(x, w)
        assert torch.equal(z, L.swiglu_linear(x, w)) if pays else z is None


@pytest.mark.gpu
@torch.inference_mode()
def test_autocast_casts(gpu):
    """In an autocast region of another dtype the products are torch's, cast as
    F.linear casts them; in one of the operands' own dtype nothing is cast."""
    x, w = _xw((8,), 64, 64, torch.bfloat16, 3)
    down = w[:, :32].contiguous()
    with torch.autocast("cuda", torch.float16):
        want = F.linear(x, w)
        assert want.dtype == torch.float16 and torch.equal(L.project(x, w), want)
        assert L.swiglu_project(x, w) is None
        z = ttt.swiglu(want[:, :32], want[:, 32:])
        assert torch.equal(ttt.swiglu_mlp(x, w, down), F.linear(z, down))
    with torch.autocast("cuda", torch.bfloat16):
        assert L._rows_for_kernel(x, w) == 8


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,glu", [
    (5, 48, 96, 0), (64, 40, 256, 1), (65, 64, 128, 0), (130, 68, 192, 1), (515, 132, 64, 0),
    (600, 36, 96, 0)])
@pytest.mark.parametrize("shift", [0, 1, 4])
@torch.inference_mode()
def test_strided_rows_and_any_output_address(gpu, M, N, K, glu, shift):
    """The C entry on a column slice of a wider x, more than MAX_ROWS rows among
    them, and on outputs at any element: the bits of the same rows packed,
    nothing written beside them."""
    wide, w = _xw((M, 3), N * (1 + glu), K, torch.bfloat16, M + N)
    x = wide[:, 1]
    want = L._run(x.contiguous(), w, M, N, glu)
    flat = torch.full((M * N + shift + 64,), 3.0, dtype=torch.bfloat16, device=gpu)
    _lib.check(_lib.lib().ttcd_linear_rows_fwd(
        x.data_ptr(), x.stride(0), w.data_ptr(), flat[shift:].data_ptr(), M, N, K, glu,
        _lib.DTYPE_BF16, _lib.stream(x)))
    assert torch.equal(flat[shift:shift + M * N].view(M, N), want)
    assert (flat[:shift] == 3.0).all() and (flat[shift + M * N:] == 3.0).all()
    if not glu:
        exact = x.double() @ w.double().T
        limit = 2.0 ** -8 * exact.abs() + K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
        assert ((want.double() - exact).abs() <= limit).all()
