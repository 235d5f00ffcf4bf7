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
from ttcd_amd import _lib, ttt

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


@pytest.mark.parametrize("B,L,rows,H,dtype", [
    (1, 5, 5, 8, torch.bfloat16), (2, 300, 257, 1024, torch.bfloat16),
    (3, 66, 64, 520, torch.float16), (1, 1030, 1023, 2048, torch.bfloat16)])
@torch.inference_mode()
def test_beta_is_the_rounded_sigmoid_of_the_rounded_product(gpu, B, L, rows, H, dtype):
    """Against 64 bits. The fp32 sum of H products is off by at most H 2^-24 of
    their magnitudes' sum, which can move the rounded product by one unit u; the
    sigmoid passes on at most a quarter of that and rounds once more."""
    g = torch.Generator().manual_seed(H + rows)
    t = torch.randn(B, L, H, generator=g).to(dtype).cuda()
    w = (torch.randn(H, generator=g) * H ** -0.5).to(dtype).cuda()
    got = ttt._beta(t, w, rows).double()
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    dot = t[:, :rows].double() @ w.double()
    size = t[:, :rows].double().abs() @ w.double().abs()
    want = torch.sigmoid(dot)
    limit = (u * dot.abs() + H * 2.0 ** -24 * size) / 4 + u * want
    assert got.shape == (B, rows) and ((got - want).abs() <= limit).all()


@pytest.mark.parametrize("B,K,C,H,dtype,with_beta", [
    (1, 2, 8, 8, torch.bfloat16, True), (2, 3, 72, 136, torch.float16, True),
    (1, 1, 64, 64, torch.bfloat16, False), (1, 2, 200, 1032, torch.bfloat16, True)])
@torch.inference_mode()
def test_transposed_update_on_whole_groups(gpu, B, K, C, H, dtype, with_beta):
    """16-byte rows and columns at the edges of the 64 x 64 tiles, bit for bit torch's
    multiply; the row stride wider than a row."""
    g = torch.Generator().manual_seed(C + H)
    pd = torch.randn(B * K * C, H + 16, generator=g).to(dtype).cuda()[:, :H]
    beta = torch.rand(B, K, C, generator=g).to(dtype).cuda() if with_beta else None
    got = ttt.proj_beta_t(pd, beta, B, K, C)
    want = pd.reshape(B, K, C, H)
    want = want * beta[..., None] if with_beta else want
    assert torch.equal(got, want.transpose(2, 3).reshape(B * K, H, C))


@pytest.mark.parametrize("nupd,nsteps,H,I,want_next", [
    (0, 1, 8, 8, False), (1, 2, 72, 136, True), (5, 4, 64, 64, True), (3, 4, 136, 1032, False)])
@torch.inference_mode()
def test_scan_on_whole_groups(gpu, nupd, nsteps, H, I, want_next):
    """Tile edges of the 16-byte scan, bit for bit torch's rounded steps."""
    g = torch.Generator().manual_seed(H + I)
    w = torch.randn(H, I, generator=g).to(torch.bfloat16).cuda()
    dw = torch.randn(nupd, H, I, generator=g).to(torch.bfloat16).cuda() if nupd else None
    steps, nxt = ttt.scan_steps(dw, w, 0.3, nsteps, want_next)
    lr = torch.tensor(0.3, dtype=torch.bfloat16, device=gpu)
    acc, ws = torch.zeros_like(w), [w]
    for j in range(nupd):
        acc = acc + dw[j]
        ws.append(w + lr * acc)
    for s_ in range(nsteps):
        assert torch.equal(steps[s_], ws[s_].t()), s_
    assert nxt is None if not want_next else torch.equal(nxt, ws[nupd])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("u", [1.0, -0.375, 250.0, 2.0 ** -10])
@torch.inference_mode()
def test_swiglu_of_every_gate(gpu, dtype, u):
    """Every bit pattern of the gate, where 1 + exp(-g) leaves fp32 and next to it
    included, against (g * (1 / (1 + exp(-g)))) * u in fp32 on the CPU: a few
    units of fp32 (2^-20) and one rounding to the dtype (its unit, or half its
    smallest subnormal); infinities and NaN where the formula has them."""
    g = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype)
    got = ttt.swiglu(g.cuda().view(64, 1024), torch.full((64, 1024), u, dtype=dtype, device=gpu))
    got = got.cpu().view(-1)
    gf = g.float()
    want = gf * (1.0 / (1.0 + torch.exp(-gf))) * u
    unit, least = (2.0 ** -8, 2.0 ** -134) if dtype == torch.bfloat16 else (2.0 ** -11, 2.0 ** -25)
    rounded = want.to(dtype)
    assert torch.equal(got.isnan(), want.isnan())
    finite = rounded.isfinite()
    assert torch.equal(got[~finite & ~want.isnan()], rounded[~finite & ~want.isnan()])
    w = want[finite].double()
    assert ((got[finite].double() - w).abs() <= (unit + 2.0 ** -20) * w.abs() + least).all()


def _mlp_weights(I=32, H=64, conv_device="cuda"):
    g = torch.Generator().manual_seed(I)
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)  # noqa: E731
    return ttt.TttMlpWeights(r(2 * I, H).cuda(), r(H, I).cuda(), r(H, H).cuda(),
                             r(I, 1, 5).to(conv_device), r(I, 1, 5).to(conv_device), r(H).cuda())


@pytest.mark.parametrize("L", [8, 40])
def test_one_chunk_refuses_what_several_do(gpu, L):
    """A prompt of one chunk reads neither the convs nor the update, and refuses the
    same calls as a longer one: a width that swiglu does not take, convs on the CPU or
    that a separate conv does not take, a gradient, an autocast region that casts the
    operands."""
    x = torch.randn(1, L, 64, generator=torch.Generator().manual_seed(L)).to(torch.bfloat16).cuda()
    call = lambda w, t=x, **kw: ttt.ttt_mlp(x, t, w, chunk=16, lr=0.3, update_every=4, **kw)  # noqa: E731
    with torch.no_grad():
        for fused in (True, False):
            with pytest.raises(_lib.TTCDError):
                call(_mlp_weights(I=20), fused=fused)
            for conv in ("kernel", "stock"):
                with pytest.raises((ValueError, RuntimeError)):
                    call(_mlp_weights(conv_device="cpu"), fused=fused, conv=conv)
        with pytest.raises(_lib.TTCDError):
            ttt.swiglu_mlp(x, _mlp_weights(I=20).gate_up, _mlp_weights(I=20).down)
        for conv, shape, dtype in (("kernel", (40, 1, 5), torch.bfloat16),
                                   ("kernel", (32, 1, 70), torch.bfloat16),
                                   ("stock", (40, 1, 5), torch.bfloat16),
                                   ("stock", (32, 1, 5), torch.float32)):
            w = _mlp_weights()
            w.conv_s = torch.ones(shape, dtype=dtype, device=gpu)
            with pytest.raises((ValueError, RuntimeError)):
                call(w, fused=False, conv=conv, scan="torch")
        down32 = _mlp_weights()
        down32.down = down32.down.float()
        for w, region in ((_mlp_weights(), torch.float16), (down32, torch.bfloat16)):
            with torch.autocast("cuda", region), pytest.raises((ValueError, RuntimeError)):
                call(w)
    w = _mlp_weights()
    with pytest.raises(RuntimeError):
        call(w, t=x.clone().requires_grad_())
    w.down.requires_grad_()
    with pytest.raises(RuntimeError):
        call(w)
    if L <= 16:  # torch's own conv takes a gradient, and its result is not read
        w = _mlp_weights()
        w.conv_s.requires_grad_()
        assert call(w, fused=False, conv="stock").shape == x.shape


@pytest.mark.parametrize("L", [8, 40])
@torch.inference_mode()
def test_empty_batches(gpu, L):
    """No sequence: an empty result by torch's operations, refused where a kernel
    would be launched."""
    x = torch.empty(0, L, 64, dtype=torch.bfloat16, device=gpu)
    call = lambda **kw: ttt.ttt_mlp(x, x, _mlp_weights(), chunk=16, lr=0.3, update_every=4, **kw)  # noqa: E731
    for kw in (dict(), dict(fused=False), dict(scan="torch")):
        with pytest.raises(ValueError):
            call(**kw)
    out = call(fused=False, conv="stock", scan="torch")
    assert out.shape == (0, L, 64) and out.dtype == torch.bfloat16


@torch.inference_mode()
def test_swiglu_output_must_hold_the_result(gpu):
    """An output of fewer rows, another dtype or device is refused before the launch;
    one of another shape or of more rows, whose first are written, is not."""
    g = torch.zeros(4, 32, dtype=torch.bfloat16, device=gpu)
    for out in (g.half(), g[:2], g[:, :16], g.cpu()):
        with pytest.raises(ValueError):
            ttt.swiglu(g, g, out=out)
    assert ttt.swiglu(g, g, out=g.view(2, 2, 32)).shape == (2, 2, 32)
    x = torch.randn(4, 32, generator=torch.Generator().manual_seed(0)).to(torch.bfloat16).to(gpu)
    more = torch.full((6, 32), 3.0, dtype=torch.bfloat16, device=gpu)
    assert torch.equal(ttt.swiglu(x, x, out=more)[:4], ttt.swiglu(x, x)) and (more[4:] == 3.0).all()


@pytest.mark.parametrize("L", [8, 16, 32, 40])
@torch.inference_mode()
def test_shapes_of_the_student_input(gpu, L):
    """Whole chunks take the student's rows in any shape; a partial one takes the
    sequences as they are, since other shapes were padded elsewhere and refused."""
    r = lambda *s: torch.randn(*s, generator=torch.Generator().manual_seed(L)).to(torch.bfloat16).cuda()  # noqa: E731
    call = lambda x, t: ttt.ttt_mlp(x, t, _mlp_weights(), chunk=16, lr=0.3, update_every=2)  # noqa: E731
    x, t = r(2, L, 64), r(2, L, 64)
    want = call(x, t)
    assert torch.equal(call(x, t.view(1, 2, L, 64)), want)
    assert torch.equal(call(x[:1], t[0]), call(x[:1], t[:1]))
    for shape in ((2 * L, 64), (2 * L * 64,), (L, 2, 64), (2, 64, L)):
        if L % 16:
            with pytest.raises(ValueError):
                call(x, t.reshape(shape))
        else:
            assert torch.equal(call(x, t.reshape(shape)), want)


@torch.inference_mode()
def test_learning_rate_weight_is_a_vector(gpu):
    """(H, 1) would give every token its rate too, one dimension deeper."""
    x = torch.randn(1, 40, 64, generator=torch.Generator().manual_seed(0)).to(torch.bfloat16).cuda()
    w = _mlp_weights()
    w.b_proj = w.b_proj[:, None]
    for scan in ("kernel", "torch"):
        with pytest.raises(ValueError):
            ttt.ttt_mlp(x, x, w, chunk=16, lr=0.3, update_every=2, scan=scan)
