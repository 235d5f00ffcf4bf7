"""The feature pass at the edges of its wavefronts (8 runs of 8 positions, 8
groups of 8 channels): chunk lengths around a run and a wavefront, channel
counts that fill no tile, every halo length, conv weights that are not 16-byte
aligned. z_hat and diff are bit for bit the oracle's conv and subtraction of
the pass's own swiglu values (which test_ipttcdv9_gpu.py holds to the oracle's
swiglu)."""
from __future__ import annotations

import pytest
import torch

from oracle import conv_ref
from ttcd_amd import ttt

pytestmark = pytest.mark.gpu


def _inputs(rows, I, K, dtype, wdt, seed, shift):
    g = torch.Generator().manual_seed(seed)
    gu = [(torch.randn(rows, 2 * I, generator=g) * 2).to(dtype).cuda() for _ in range(2)]
    w = []
    for _ in range(2):
        flat = (torch.randn(I * K + shift, generator=g) * 0.5).to(wdt).cuda()
        w.append(flat[shift:].view(I, K))
    return gu, w


@pytest.mark.parametrize("B,nchunk,C,I,K,dtype,wdt,shift", [
    (1, 2, 7, 8, 5, torch.bfloat16, torch.bfloat16, 0),
    (2, 3, 8, 72, 8, torch.bfloat16, torch.bfloat16, 0),
    (1, 2, 63, 64, 2, torch.float16, torch.float16, 0),
    (1, 3, 64, 56, 5, torch.bfloat16, torch.bfloat16, 1),   # weights off alignment
    (2, 2, 65, 136, 7, torch.bfloat16, torch.float32, 1),
    (1, 2, 200, 64, 3, torch.float16, torch.bfloat16, 3),
    (1, 2, 130, 64, 1, torch.bfloat16, torch.bfloat16, 0),
])
@torch.inference_mode()
def test_features_at_tile_edges(gpu, B, nchunk, C, I, K, dtype, wdt, shift):
    rows = B * nchunk * C
    (gu_t, gu_s), (w_t, w_s) = _inputs(rows, I, K, dtype, wdt, C + I + K, shift)
    z, zh, diff = ttt.ttt_features(gu_t, gu_s, w_t, w_s, B, nchunk, C)
    zr = ttt.swiglu(gu_s[:, :I], gu_s[:, I:])
    assert torch.equal(z, ttt.swiglu(gu_t[:, :I], gu_t[:, I:]))
    want_zh = conv_ref.dwconv_c(zr.cpu().view(-1, C, I), w_s.cpu()).view(B, nchunk, C, I)
    tgt = conv_ref.dwconv_c(z.cpu().view(-1, C, I), w_t.cpu()).view(B, nchunk, C, I)
    assert torch.equal(zh.cpu(), want_zh.reshape(-1, I))
    want = (tgt[:, :-1].float() - want_zh[:, :-1].float()).to(dtype).reshape(-1, I)
    assert torch.equal(diff.cpu(), want)


@pytest.mark.parametrize("B,tokens,C,I,ct,cs", [
    (1, 100, 64, 64, True, True), (2, 129, 64, 72, True, False), (3, 65, 32, 64, False, True),
    (2, 128, 64, 64, True, True), (1, 4097, 4096, 64, True, True), (2, 50, 7, 8, False, False)])
@torch.inference_mode()
def test_features_of_tokens_equal_the_padded_pass(gpu, B, tokens, C, I, ct, cs):
    """Sequences that are not whole chunks: the features of the zero-padded rows,
    bit for bit, from unpadded rows with nothing after the last one needed."""
    nchunk, K = -(-tokens // C), 5
    upd = (nchunk - 1) * C
    (gu_t, gu_s), (w_t, w_s) = _inputs(B * tokens, I, K, torch.bfloat16, torch.bfloat16,
                                       tokens + I, 0)
    w_t, w_s = w_t if ct else None, w_s if cs else None
    z, zh, diff = ttt._features_tokens(gu_t, gu_s[:(B - 1) * tokens + upd], w_t, w_s, B, tokens, C)
    pad = [torch.nn.functional.pad(v.view(B, tokens, 2 * I), (0, 0, 0, nchunk * C - tokens))
           .reshape(-1, 2 * I) for v in (gu_t, gu_s)]
    wz, wzh, wdiff = ttt.ttt_features(pad[0], pad[1], w_t, w_s, B, nchunk, C)
    assert torch.equal(z, wz.view(B, nchunk * C, I)) and torch.equal(diff, wdiff)
    assert torch.equal(zh, wzh.view(B, nchunk * C, I)[:, :upd].reshape(-1, I))
