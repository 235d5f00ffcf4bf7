"""Cached prefills split over keys (ttcd_attn_kv_workspace_bytes > 0).

The parts fold the same scores in the same tiles as the whole call, each
against its own reference max, and are added in fp32; so a split call is held
to the whole call (the C entry without a workspace, itself held to the oracle
by test_kv_attn_gpu.py) by the rounding of the probabilities and of the
result: each probability is rounded to the input dtype in both calls, against
different references, so a row's output may move by 2 u sum_j p_j |v_j| (u the
dtype's unit roundoff) plus one unit of the result's own rounding, and its LSE
only by fp32 sums (of up to 8192 terms, 1e-5)."""
from __future__ import annotations

import pytest
import torch

from conftest import make_qkv
from ttcd_amd import (_lib, band_attn, fused_dual_window_attn, lse_dual_window_attn,
                      window_attn)

DT = {torch.bfloat16: _lib.DTYPE_BF16, torch.float16: _lib.DTYPE_F16}


def _bytes(B, Tq, Tk, H, HK, D, lo, mid, hi, rescale=8.0):
    return _lib.lib().ttcd_attn_kv_workspace_bytes(B, Tq, Tk, H, HK, D, lo, mid, hi, rescale)


def test_what_is_split():
    one = 300 * 16 * 129 * 4  # bytes of one part
    n = _bytes(1, 300, 8491, 16, 8, 128, 0, 8192, 8192)
    assert n % one == 0 and 2 <= n // one <= 32
    assert _bytes(1, 300, 8491, 16, 8, 128, 0, 4096, -1) % one == 0
    for call in ((1, 2048, 10239, 15, 5, 64, 0, 4096, 8192), (1, 4096, 12287, 4, 2, 64, 0, 4096, 8192)):
        assert _bytes(*call) > 0, call
    for call in ((1, 8491, 8491, 16, 8, 128, 0, 8192, 8192),    # not cached
                 (1, 300, 4600, 16, 8, 128, 0, 4224, 4224),     # 4 KiB of keys, as one sweep
                 (1, 8000, 16191, 16, 8, 128, 0, 8192, 8192),   # fills the GPU
                 # rows with a part of their window: the unsplit sweeps are the shorter
                 (1, 11186, 27569, 4, 4, 128, 0, 27569, 27569),
                 # one part with nearly all of the window
                 (2, 4301, 9079, 4, 2, 64, 0, 7168, 9079), (3, 910, 9507, 15, 5, 64, 0, 8064, 9507),
                 (1, 300, 8491, 16, 7, 128, 0, 8192, 8192),     # not a call
                 (1, 300, 8491, 16, 8, 96, 0, 8192, 8192),
                 (1, 300, 8491, 16, 8, 128, 4, 4, 8)):
        assert _bytes(*call) == 0, call
    assert _bytes(1, 300, 8491, 16, 8, 128, 0, 8192, 8192, 0.0) == 0  # exact running max


def _whole(q, k, v, lo, mid, hi, dual):
    B, T, H, D = q.shape
    ot, os_ = torch.empty_like(q), torch.empty_like(q)
    lt, ls = (torch.empty(B, H, T, device=q.device) for _ in range(2))
    st = [_lib.strides4(x.stride()) for x in (q, k, v, ot)]
    L = _lib.lib()
    shape = (B, T, k.shape[1], H, k.shape[2], D)
    stream = torch.cuda.current_stream().cuda_stream
    if dual:
        _lib.check(L.ttcd_dual_window_attn_kv_fwd(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), ot.data_ptr(), os_.data_ptr(),
            lt.data_ptr(), ls.data_ptr(), *shape, *st, hi, mid, D ** -0.5, 8.0, DT[q.dtype],
            stream))
        return ot, os_, lt, ls
    _lib.check(L.ttcd_band_attn_kv_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), ot.data_ptr(), lt.data_ptr(), *shape, *st, lo,
        hi, D ** -0.5, 8.0, DT[q.dtype], stream))
    return ot, lt


def _close(got, want, bound, dtype, what):
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    g, w = got.float(), want.float()
    limit = 2 * u * bound + u * w.abs() + 1e-6
    worst = ((g - w).abs() / limit).max().item()
    assert worst <= 1.0, (what, worst)


@pytest.mark.gpu
@pytest.mark.parametrize("B,Tq,Tk,H,HK,D,wt,ws,dtype", [
    (1, 1, 8192, 16, 8, 128, 8192, 4096, torch.bfloat16),     # one token, two heads a wavefront
    (1, 300, 8491, 16, 8, 128, 8192, 4096, torch.bfloat16),
    (2, 65, 6001, 4, 4, 128, -1, 33, torch.float16),          # full causal, near part of a tile
    (1, 129, 9000, 15, 5, 64, 8192, 8064, torch.bfloat16),    # far part of two tiles
    (1, 70, 5000, 4, 2, 64, 4999, 4998, torch.float16),       # far part of one key
    (3, 7, 16390, 8, 2, 128, 16384, 8192, torch.bfloat16),
    (1, 200, 5100, 8, 1, 64, 6000, 5100, torch.bfloat16),     # windows past the keys: no far part
    # 24 pairs of part and head, dealt to the XCDs from one later every round, and with
    # whole windows in runs
    (1, 1454, 5526, 4, 4, 64, -1, 1000, torch.bfloat16),
    (1, 2599, 8674, 4, 4, 128, 6000, 3000, torch.float16),
])
@torch.inference_mode()
def test_split_calls_match_the_whole_call(gpu, B, Tq, Tk, H, HK, D, wt, ws, dtype):
    qf, k, v = make_qkv(batch=B, seqlen=Tk, heads=H, kv_heads=HK, head_dim=D, dtype=dtype,
                        seed=Tq + Tk)
    q = qf[:, Tk - Tq:]
    k = torch.stack([k, v], 2).flatten(2, 3)[:, :, :HK]  # strided keys
    hi = wt if wt > 0 else Tk
    assert _bytes(B, Tq, Tk, H, HK, D, 0, ws, hi) > 0 and _bytes(B, Tq, Tk, H, HK, D, 0, hi, hi) > 0
    mean_abs_v = window_attn(q, k, v.abs(), hi)  # sum_j p_j |v_j|, to its own rounding
    got = fused_dual_window_attn(q, k, v, wt, ws, return_lse=True)
    want = _whole(q, k, v, 0, ws, hi, True)
    near = window_attn(q, k, v.abs(), ws)
    for name, g, w, b in (("teacher", got[0], want[0], mean_abs_v), ("student", got[1], want[1], near)):
        _close(g, w, 1.02 * b.float(), dtype, name)
    assert (got[2] - want[2]).abs().max() <= 1e-5 and (got[3] - want[3]).abs().max() <= 1e-5
    o, lse = window_attn(q, k, v, wt, return_lse=True)
    wo, wl = _whole(q, k, v, 0, hi, hi, False)
    _close(o, wo, 1.02 * mean_abs_v.float(), dtype, "window")
    assert (lse - wl).abs().max() <= 1e-5


@pytest.mark.gpu
@torch.inference_mode()
def test_split_call_under_graph_capture(gpu):
    qf, k, v = make_qkv(batch=1, seqlen=8300, heads=16, kv_heads=8, head_dim=128, seed=5)
    q = qf[:, -40:].contiguous()
    want = window_attn(q, k, v, 8192)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = window_attn(q, k, v, 8192)
    for _ in range(3):
        out.fill_(7.0)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.gpu
@pytest.mark.parametrize("H,HK,D,dtype", [
    (16, 8, 128, torch.bfloat16), (4, 4, 128, torch.float16), (15, 5, 64, torch.bfloat16),
    (4, 2, 64, torch.float16)])
@pytest.mark.parametrize("Tq,Tk,ws,near,far", [
    (40, 8231, 1000, 5.0, 55.0), (40, 8231, 1000, 5.0, 95.0), (40, 8231, 1000, 5.0, 105.0),
    (40, 8231, 1000, 5.0, 205.0), (40, 8231, 4096, 150.0, -50.0),
    # rows without a far key among rows with some, every score far below zero
    (200, 9000, 8900, -150.0, -150.0)])
@torch.inference_mode()
def test_near_and_far_scores_far_apart(gpu, Tq, Tk, ws, near, far, H, HK, D, dtype):
    """Scores offset by `near` nats within the student window and by `far` beyond it, up to
    200 apart, past what exp spans in fp32: the student is its own window's
    softmax however large the far scores are. An LSE of size |L| is a product and
    sums in fp32: eight units of L in either call."""
    q, k, v = make_qkv(batch=1, seqlen=Tk, heads=H, kv_heads=HK, head_dim=D, dtype=dtype,
                       seed=Tk + ws)
    q = q[:, Tk - Tq:].clone()
    q[..., 0] = 16.0
    reach = Tk - Tq - ws + 1 if near != far else 0  # keys no row's student window holds
    k[..., 0] = near / (16.0 * D ** -0.5)
    k[:, :reach, :, 0] = far / (16.0 * D ** -0.5)
    assert _bytes(1, Tq, Tk, H, HK, D, 0, ws, Tk) > 0
    got = fused_dual_window_attn(q, k, v, -1, ws, return_lse=True)
    want = _whole(q, k, v, 0, ws, Tk, True)
    assert all(torch.isfinite(x).all() for x in got)
    if near != far:
        gap = want[2] - want[3]
        assert (gap - max(far - near, 0.0)).abs().max() < 12.0  # the keys' own spread
    for name, g, w, W in (("teacher", got[0], want[0], Tk), ("student", got[1], want[1], ws)):
        _close(g, w, 1.02 * window_attn(q, k, v.abs(), W).float(), dtype, name)
    for g, w in ((got[2], want[2]), (got[3], want[3])):
        assert ((g - w).abs() <= 1e-5 + 2.0 ** -21 * w.abs()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("B,Tq,Tk,H,HK,D,wt,ws", [
    (1, 300, 8491, 16, 8, 128, 8192, 4736), (2, 33, 5000, 15, 5, 64, -1, 4736)])
@torch.inference_mode()
def test_rows_that_are_not_split_have_the_bits_of_the_whole_prompt(gpu, B, Tq, Tk, H, HK, D, wt, ws):
    """split_keys=False on calls that would be split: the last rows of the call on the
    whole prompt, bit for bit; the LSE variant's student likewise."""
    qf, k, v = make_qkv(batch=B, seqlen=Tk, heads=H, kv_heads=HK, head_dim=D, seed=Tk)
    q = qf[:, Tk - Tq:]
    hi = wt if wt > 0 else Tk
    for lo, mid, top in ((0, ws, hi), (0, hi, hi), (0, ws, ws), (16, hi, hi)):
        assert _bytes(B, Tq, Tk, H, HK, D, lo, mid, top) > 0
    kw = dict(return_lse=True, split_keys=False)
    for got, want in zip(fused_dual_window_attn(q, k, v, wt, ws, **kw),
                         fused_dual_window_attn(qf, k, v, wt, ws, return_lse=True)):
        rows = want[..., Tk - Tq:] if want.dim() == 3 else want[:, Tk - Tq:]
        assert torch.equal(got, rows)
    for lo, top in ((0, hi), (16, hi)):
        o, lse = band_attn(q, k, v, lo, top, **kw)
        wo, wl = band_attn(qf, k, v, lo, top, return_lse=True)
        assert torch.equal(o, wo[:, Tk - Tq:]) and torch.equal(lse, wl[..., Tk - Tq:])
    student = window_attn(q, k, v, ws, split_keys=False)
    assert torch.equal(lse_dual_window_attn(q, k, v, wt, ws)[1], student)
    assert torch.equal(window_attn(q[:1], k[:1], v[:1], ws, split_keys=False), student[:1])
