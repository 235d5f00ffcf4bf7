"""The work a user of this package has it do, as cases that can be timed and compared.

Each case is one call (or one short sequence of calls) of the package's public
entry points on inputs made from a seed. Sizes are those of the repository's
own model configurations, tests and benchmark; `draw` gives more of the same
ranges. `exact` is the same mathematics in plain torch, in 64 bits.

Kinds
  dual      fused_dual_window_attn: the attention of a TTT layer's prefill
  window    window_attn: the attention of a plain layer, also onto a cache (Tk > Tq)
  lse       lse_dual_window_attn: the log-sum-exp variant of `dual`
  varlen    fused_dual_window_attn_varlen: packed sequences
  conv      causal_dwconv_x: the chunk-local conv of the TTT MLP
  prologue  qk_norm_rope on views of one fused projection output
  epilogue  fused_attn_epilogue: o_proj of both outputs, then both residual norms
  ttt       ttt_mlp: the TTT MLP's prefill
  prefill   IPTTCDv9Prefill.forward, whole or in chunks over a cache; returns logits
"""
import math

import torch
import torch.nn.functional as F

import ttcd_amd
from ttcd_amd import ipttcdv9, ttt

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
DEV = "cuda"


def listed():
    return [
        # the smallest layer of the test suite: a short prompt, where launch and
        # host latency count
        _attn("dual", name="dual-short", B=1, Tq=2048, Tk=2048, Hq=4, Hkv=2, D=64, wt=512, ws=256),
        # the benchmark's headline: one TTT layer of a 64K prefill, Qwen3-0.6B shape
        _attn("dual", name="dual-qwen3-64k", B=1, Tq=65536, Tk=65536, Hq=16, Hkv=8, D=128,
              wt=8192, ws=4096, lse=True),
        # the same for the SmolLM2-360M shape: head size 64, three query heads per K/V head
        _attn("dual", name="dual-smollm2-64k", B=1, Tq=65536, Tk=65536, Hq=15, Hkv=5, D=64,
              wt=8192, ws=4096),
        # an ordinary batch of ragged prompts in fp16
        _attn("dual", name="dual-f16-ragged", B=2, Tq=5003, Tk=5003, Hq=16, Hkv=8, D=128,
              wt=2048, ws=1024, dtype="f16"),
        # a follow-up prompt of 300 tokens prefilled onto a full 8192-token window
        _attn("window", name="window-cached", B=1, Tq=300, Tk=8491, Hq=16, Hkv=8, D=128, wt=8192),
        # the LSE variant at the batch sweep's length
        _attn("lse", name="lse-16k", B=1, Tq=16384, Tk=16384, Hq=16, Hkv=8, D=128, wt=8192,
              ws=4096),
        # a packed batch of sequences of mixed length
        dict(kind="varlen", name="varlen-packed", total=12345, nseq=9, Hq=15, Hkv=5, D=64, wt=2048,
             ws=1024, dtype="bf16", lse=False, exact_max=False),
        # the TTT MLP's conv over a 64K prefill
        dict(kind="conv", name="conv-64k", N=16, C=4096, D=3072, K=5, dtype="bf16"),
        # the attention prologue of a 16K prefill
        dict(kind="prologue", name="prologue-16k", B=1, T=16384, Hq=16, Hkv=8, D=128, offset=0,
             norm=True, dtype="bf16"),
        # the attention epilogue of one TTT layer, a ragged prompt
        dict(kind="epilogue", name="epilogue-ragged", B=1, T=10007, H=1024, A=2048, dtype="bf16"),
        # the TTT MLP of a prompt that is not a whole number of chunks
        dict(kind="ttt", name="ttt-mlp-24k", B=1, T=24000, H=1024, I=3072, chunk=4096, every=16,
             K=5, dtype="bf16"),
        # a whole prefill: four layers of the Qwen3-0.6B shape, the first a TTT layer
        dict(kind="prefill", name="prefill-4-layers", B=1, T=4500, layers=4, chunk=0, keep=8),
    ]


def _attn(kind, *, B, Tq, Tk, Hq, Hkv, D, wt, ws=0, dtype="bf16", lse=False, exact_max=False,
          name=None):
    case = dict(kind=kind, B=B, Tq=Tq, Tk=Tk, Hq=Hq, Hkv=Hkv, D=D, wt=wt, ws=ws, dtype=dtype,
                lse=lse, exact_max=exact_max)
    return case if name is None else dict(case, name=name)


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("dual", "dual", "window", "window", "lse", "varlen", "conv", "conv",
                       "prologue", "epilogue", "ttt", "ttt", "prefill", "prefill"))
    dtype = rng.choice(("bf16", "bf16", "bf16", "f16"))
    Hq, Hkv, D = rng.choice(((16, 8, 128), (16, 8, 128), (15, 5, 64), (4, 2, 64), (8, 2, 128),
                             (4, 4, 128)))
    wt, ws = rng.choice(((8192, 4096), (8192, 4096), (8192, 7168), (8192, 8064), (2048, 1024),
                         (16384, 8192), (512, 256), (-1, 4096)))
    if kind in ("dual", "window", "lse"):
        B = rng.choice((1, 1, 1, 2, 3))
        Tq = _log_int(rng, 200, 28000 // B if wt < 0 or wt > 8192 else 60000 // B)
        if kind == "window":
            # a call onto a cache: one token up to a prefill chunk, over a full window
            Tq = _log_int(rng, 1, 16384 // B)
            cached = rng.choice((0, wt - 1 if wt > 0 else 16383, _log_int(rng, 100, 16383)))
        else:
            cached = rng.choice((0, 0, 0, min(max(wt, 1024), 8192) - 1))
        Tk = Tq + min(cached, 32768)
        ws = min(ws, Tk - 1) if kind == "dual" else min(ws, max(wt if wt > 0 else Tk, 2) - 1)
        return _attn(kind, B=B, Tq=Tq, Tk=Tk, Hq=Hq, Hkv=Hkv, D=D, wt=wt,
                     ws=0 if kind == "window" else max(ws, 1), dtype=dtype,
                     lse=kind != "lse" and rng.random() < 0.4,
                     exact_max=rng.random() < 0.2)
    if kind == "varlen":
        return dict(kind=kind, total=_log_int(rng, 300, 24000 if wt < 0 or wt > 8192 else 40000), nseq=rng.randint(1, 24), Hq=Hq,
                    Hkv=Hkv, D=D, wt=wt, ws=ws, dtype=dtype, lse=rng.random() < 0.4,
                    exact_max=rng.random() < 0.2)
    if kind == "conv":
        C = rng.choice((4096, 2048, 256, rng.randint(1, 4500)))
        D = rng.choice((3072, 2560, 256, rng.randint(1, 3100), 8 * rng.randint(1, 400)))
        dt = rng.choice(("bf16", "bf16", "f16", "f32"))
        rows = _log_int(rng, 64, 65536 if dt != "f32" else 32768)
        return dict(kind=kind, N=max(1, rows // C), C=C, D=D, K=rng.choice((5, 5, 5, 4, 3, 2, 7, 9)),
                    dtype=dt)
    if kind == "prologue":
        return dict(kind=kind, B=rng.choice((1, 1, 2)), T=_log_int(rng, 1, 32768), Hq=Hq, Hkv=Hkv,
                    D=D, offset=rng.choice((0, 0, rng.randint(1, 8192))), norm=rng.random() < 0.8,
                    dtype=dtype)
    if kind == "epilogue":
        H, A = rng.choice(((1024, 2048), (960, 960), (1024, 2048), (256, 512), (2048, 2048)))
        return dict(kind=kind, B=rng.choice((1, 1, 2)), T=_log_int(rng, 1, 32768), H=H, A=A,
                    dtype=dtype)
    if kind == "ttt":
        H, I = rng.choice(((1024, 3072), (1024, 3072), (960, 2560), (256, 768)))
        chunk = rng.choice((4096, 4096, 2048, 256))
        B = rng.choice((1, 1, 2))
        top = min(49152, chunk * 24) // B
        T = rng.choice((_log_int(rng, chunk, top), chunk * max(1, _log_int(rng, chunk, top) // chunk)))
        return dict(kind=kind, B=B, T=T, H=H, I=I, chunk=chunk, every=rng.choice((16, 16, 4)),
                    K=rng.choice((5, 5, 4)), dtype=dtype)
    B = rng.choice((1, 1, 2))
    T = _log_int(rng, 1, 9000 // B)
    return dict(kind="prefill", B=B, T=T, layers=rng.randint(1, 4),
                chunk=rng.choice((0, 0, max(1, T // rng.randint(1, 4)))), keep=rng.choice((1, 8)))


# ------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, dtype=torch.bfloat16, std=1.0):
    x = torch.randn(*shape, generator=g, device=DEV, dtype=dtype)
    return x if std == 1.0 else x.mul_(std)


def _lengths(case):
    """nseq sequence lengths that add up to `total`, very unequal."""
    n, total = case["nseq"], case["total"]
    cuts = sorted(total * (i * i + i % 3) // (n * n + 3) for i in range(1, n))
    edges = [0] + cuts + [total]
    return [b - a for a, b in zip(edges, edges[1:])]


def _model_cfg(case):
    return dict(ipttcdv9.QWEN3_06B_SWA8K, num_hidden_layers=case["layers"], ttt_layers=[0],
                ttt_teacher_conv_init="random", ttt_student_conv_init="random")


def _qkv(case, g):
    """q and k as the prologue leaves them, v a view of the fused projection's output."""
    B, Tq, Tk, Hq, Hkv, D = (case[n] for n in ("B", "Tq", "Tk", "Hq", "Hkv", "D"))
    dt = DTYPES[case["dtype"]]
    q = _randn(g, B, Tq, Hq, D, dtype=dt)
    k = _randn(g, B, Tk, Hkv, D, dtype=dt)
    if Tk > Tq:
        return q, k, _randn(g, B, Tk, Hkv, D, dtype=dt)
    return q, k, _randn(g, B, Tk, 2 * Hkv, D, dtype=dt)[:, :, Hkv:]


def _packed(case, g):
    dt, total = DTYPES[case["dtype"]], case["total"]
    q = _randn(g, total, case["Hq"], case["D"], dtype=dt)
    k = _randn(g, total, case["Hkv"], case["D"], dtype=dt)
    v = _randn(g, total, case["Hkv"], case["D"], dtype=dt)
    return q, k, v


def _conv(case, g):
    dt = DTYPES[case["dtype"]]
    x = _randn(g, case["N"], case["C"], case["D"], dtype=dt)
    return x, _randn(g, case["D"], case["K"], dtype=dt, std=0.5)


def _prologue(case, g):
    B, T, Hq, Hkv, D = (case[n] for n in ("B", "T", "Hq", "Hkv", "D"))
    dt = DTYPES[case["dtype"]]
    qkv = _randn(g, B, T, (Hq + 2 * Hkv) * D, dtype=dt, std=0.64)
    q = qkv[..., :Hq * D].view(B, T, Hq, D)
    k = qkv[..., Hq * D:(Hq + Hkv) * D].view(B, T, Hkv, D)
    w = None
    if case["norm"]:
        w = [1 + _randn(g, D, dtype=dt, std=0.1) for _ in range(2)]
    return q, k, w


def _epilogue(case, g):
    B, T, H, A = (case[n] for n in ("B", "T", "H", "A"))
    dt = DTYPES[case["dtype"]]
    both = _randn(g, 2, B, T, A, dtype=dt)  # the attention call's two outputs
    res = _randn(g, B, T, H, dtype=dt)
    return both, res, _randn(g, H, A, dtype=dt, std=0.02), 1 + _randn(g, H, dtype=dt, std=0.1)


def _ttt(case, g):
    B, T, H, I, K = (case[n] for n in ("B", "T", "H", "I", "K"))
    dt = DTYPES[case["dtype"]]
    both = _randn(g, 2, B, T, H, dtype=dt)  # the epilogue's two normalised outputs
    w = dict(gate_up=_randn(g, 2 * I, H, dtype=dt, std=0.02),
             down=_randn(g, H, I, dtype=dt, std=0.02),
             ttt_proj=torch.diag(_randn(g, H, dtype=dt, std=0.02)),
             conv_t=_randn(g, I, 1, K, dtype=dt, std=0.02),
             conv_s=_randn(g, I, 1, K, dtype=dt, std=0.02),
             b_proj=_randn(g, H, dtype=dt, std=0.02))
    w["conv_t"][:, 0, K - 1] += 1.0
    return both, w


class _Norm:
    def __init__(self, weight, eps):
        self.weight, self.bias, self.eps = weight, None, eps


class _Linear:
    def __init__(self, weight):
        self.weight, self.bias = weight, None


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind in ("dual", "window", "lse"):
        return dict(case=case, qkv=_qkv(case, g))
    if kind == "varlen":
        lens = _lengths(case)
        cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).to(DEV)
        return dict(case=case, qkv=_packed(case, g), cu=cu, longest=max(lens))
    if kind == "conv":
        return dict(case=case, xw=_conv(case, g))
    if kind == "prologue":
        q, k, w = _prologue(case, g)
        inv = ttcd_amd.rope_inv_freq(case["D"], 1000000.0, DEV)
        cos, sin = ttcd_amd.rope_tables(inv, case["T"] + case["offset"], q.dtype)
        return dict(case=case, q=q, k=k, w=w or (None, None), cos=cos, sin=sin)
    if kind == "epilogue":
        both, res, w, nw = _epilogue(case, g)
        return dict(case=case, both=both, res=res, proj=_Linear(w), norm=_Norm(nw, 1e-6))
    if kind == "ttt":
        both, w = _ttt(case, g)
        return dict(case=case, both=both, w=ttt.TttMlpWeights(**w))
    cfg = _model_cfg(case)
    model = ipttcdv9.IPTTCDv9Prefill(cfg, ipttcdv9.init_weights(cfg, torch.device(DEV, 0), seed=seed))
    model.tables(case["T"])
    ids = torch.randint(0, cfg["vocab_size"], (case["B"], case["T"]), generator=g, device=DEV)
    return dict(case=case, model=model, ids=ids)


@torch.inference_mode()
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "dual":
        return ttcd_amd.fused_dual_window_attn(*state["qkv"], case["wt"], case["ws"],
                                               return_lse=case["lse"],
                                               exact_max=case["exact_max"])
    if kind == "window":
        return ttcd_amd.window_attn(*state["qkv"], case["wt"], return_lse=case["lse"],
                                    exact_max=case["exact_max"])
    if kind == "lse":
        return ttcd_amd.lse_dual_window_attn(*state["qkv"], case["wt"], case["ws"],
                                             exact_max=case["exact_max"])
    if kind == "varlen":
        return ttcd_amd.fused_dual_window_attn_varlen(
            *state["qkv"], state["cu"], state["longest"], case["wt"], case["ws"],
            return_lse=case["lse"], exact_max=case["exact_max"])
    if kind == "conv":
        return ttcd_amd.causal_dwconv_x(*state["xw"])
    if kind == "prologue":
        return ttcd_amd.qk_norm_rope(state["q"], state["k"], *state["w"], 1e-6, state["cos"],
                                     state["sin"], case["offset"])
    if kind == "epilogue":
        return ttcd_amd.fused_attn_epilogue(state["proj"], state["norm"], state["both"][0],
                                            state["both"][1], state["res"])
    if kind == "ttt":
        return ttt.ttt_mlp(state["both"][0], state["both"][1], state["w"], chunk=case["chunk"],
                           lr=0.3, update_every=case["every"])
    ids, model, n = state["ids"], state["model"], case["chunk"]
    if not n:
        return model.forward(ids, logits_to_keep=case["keep"])
    cache = ttcd_amd.IPTTCDv9Cache()
    return [model.forward(ids[:, a:a + n], logits_to_keep=case["keep"], cache=cache)
            for a in range(0, ids.shape[1], n)]


# --------------------------------------------------------------------- work

def _pairs(Tq, Tk, W):
    """Visible (query, key) pairs of the last Tq of Tk positions under window W."""
    def upto(n):
        return n * (n + 1) // 2 if W < 0 or n <= W else W * (W + 1) // 2 + (n - W) * W
    return upto(Tk) - upto(Tk - Tq)


def _ttt_flops(B, T, H, I, chunk):
    n = -(-T // chunk)
    upd = B * (n - 1) * chunk
    return (8 * B * T * H * I + 2 * B * T * H * I       # gate|up of both, output
            + (4 * upd * H * I + 2 * I * H * H if n > 1 else 0))  # projection, update


def work(case):
    """Each input read once, each output written once, and the operations of the
    algorithm (attention: the teacher's band, of which the student's is a part)."""
    kind = case["kind"]
    e = 4 if case.get("dtype") == "f32" else 2
    if kind in ("dual", "window", "lse"):
        B, Tq, Tk, Hq, Hkv, D = (case[n] for n in ("B", "Tq", "Tk", "Hq", "Hkv", "D"))
        outs = 1 if kind == "window" else 2
        seen = Tk if case["wt"] < 0 else min(Tk, Tq + case["wt"] - 1)
        return {"bytes": e * B * D * ((1 + outs) * Tq * Hq + 2 * seen * Hkv)
                + (4 * outs * B * Tq * Hq if case["lse"] else 0),
                "flops": 4 * B * Hq * D * _pairs(Tq, Tk, case["wt"])}
    if kind == "varlen":
        total, Hq, Hkv, D = (case[n] for n in ("total", "Hq", "Hkv", "D"))
        return {"bytes": e * total * D * (3 * Hq + 2 * Hkv) + (8 * total * Hq if case["lse"] else 0),
                "flops": 4 * Hq * D * sum(_pairs(n, n, case["wt"]) for n in _lengths(case))}
    if kind == "conv":
        n = case["N"] * case["C"] * case["D"]
        return {"bytes": e * (2 * n + case["D"] * case["K"]), "flops": 2 * n * case["K"]}
    if kind == "prologue":
        B, T, D, heads = case["B"], case["T"], case["D"], case["Hq"] + case["Hkv"]
        return {"bytes": e * (2 * B * T * heads * D + T * D), "flops": 8 * B * T * heads * D}
    if kind == "epilogue":
        rows, H, A = case["B"] * case["T"], case["H"], case["A"]
        return {"bytes": e * (2 * rows * A + A * H + 4 * rows * H + H), "flops": 4 * rows * A * H}
    if kind == "ttt":
        B, T, H, I = (case[n] for n in ("B", "T", "H", "I"))
        return {"bytes": e * (3 * B * T * H + 3 * I * H + H * H + 2 * I * case["K"] + H),
                "flops": _ttt_flops(B, T, H, I, case["chunk"])}
    c = _model_cfg(case)
    B, T, L = case["B"], case["T"], case["layers"]
    H, I, V, D = c["hidden_size"], c["intermediate_size"], c["vocab_size"], c["head_dim"]
    Hq, Hkv, W, C = c["num_heads"], c["num_kv_heads"], c["window_size"], c["ttt_chunk"]
    step = case["chunk"] or T
    flops = weights = logits = 0
    for a in range(0, T, step):
        n = min(step, T - a)
        tok = B * n
        plain = 2 * tok * H * (2 * Hq + 2 * Hkv) * D + 4 * B * Hq * D * _pairs(n, a + n, W)
        flops += L * plain + (L - 1) * 6 * tok * H * I
        flops += _ttt_flops(B, n, H, I, C) + 2 * tok * Hq * D * H if n >= C else 6 * tok * H * I
        keep = min(case["keep"], n)
        flops += 2 * B * keep * H * V
        logits += B * keep * V
    weights = L * H * (2 * Hq + 2 * Hkv) * D + L * 3 * H * I + V * H
    return {"bytes": 2 * (weights + B * T * H + logits) + 8 * B * T, "flops": flops}


def tolerance(case):
    """About four times what each path is off from `exact` on an MI355X (attention
    2.4e-3 in bf16 and 2.7e-4 in f16, prologue 2.7e-3, epilogue 2.1e-3, TTT MLP
    3.8e-3, prefill logits 1.0e-2): the 16-bit rounding of the results and of the
    values the path itself rounds (the probabilities, a block's hidden states).
    The conv has one fixed order of accumulation and is compared bit for bit."""
    kind = case["kind"]
    if kind == "conv":
        return "exact"
    bf16 = case.get("dtype", "bf16") == "bf16"
    if kind == "prefill":
        return {"rel": 0.03}
    if kind == "ttt":
        return {"rel": 0.015 if bf16 else 0.002}
    return {"rel": 0.01 if bf16 else 0.0013}


# ------------------------------------------------------------ in 64 bits

def _attention64(q, k, v, windows):
    """For each window W: (output, LSE) of the last Tq of Tk positions, in blocks
    of query rows against the keys their widest window reaches. q (Tq, Hq, D)."""
    Tq, Hq, D = q.shape
    Tk, Hkv = k.shape[0], k.shape[1]
    G, scale = Hq // Hkv, D ** -0.5
    q, k, v = (x.double().transpose(0, 1) for x in (q, k, v))  # (H, T, D)
    widest = Tk if any(W < 0 for W in windows) else max(windows)
    step = max(64, min(1024, (1 << 28) // (Hq * min(Tk, widest + 1024))))
    outs = [(torch.empty(Hq, Tq, D, dtype=torch.float64, device=q.device),
             torch.empty(Hq, Tq, dtype=torch.float64, device=q.device)) for _ in windows]
    for r0 in range(0, Tq, step):
        r1 = min(Tq, r0 + step)
        i0, i1 = Tk - Tq + r0, Tk - Tq + r1
        j0 = max(0, i0 - widest + 1)
        kk = k[:, j0:i1].transpose(1, 2).contiguous()
        vv = v[:, j0:i1].contiguous()
        s = torch.bmm(q[:, r0:r1].reshape(Hkv, G * (r1 - r0), D), kk).mul_(scale)
        s = s.view(Hkv, G, r1 - r0, i1 - j0)
        d = torch.arange(i0, i1, device=q.device)[:, None] - torch.arange(j0, i1, device=q.device)
        s.masked_fill_(d < 0, -math.inf)
        for (o, lse), W in sorted(zip(outs, windows), key=lambda x: -(x[1] if x[1] > 0 else Tk)):
            if W > 0:
                s.masked_fill_(d >= W, -math.inf)
            m = s.amax(-1, keepdim=True)
            p = (s - m).exp_()
            tot = p.sum(-1, keepdim=True)
            o[:, r0:r1] = (torch.bmm(p.view(Hkv, -1, i1 - j0), vv).view(Hkv, G, r1 - r0, D)
                           / tot).reshape(Hq, r1 - r0, D)
            lse[:, r0:r1] = (m + tot.log()).reshape(Hq, r1 - r0)
    return [(o.transpose(0, 1), lse) for o, lse in outs]


def _norm64(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _rope64(x, offset, base=1000000.0):
    D, T = x.shape[-1], x.shape[-3]
    inv = base ** (-torch.arange(0, D, 2, device=x.device, dtype=torch.float64) / D)
    f = torch.outer(torch.arange(offset, offset + T, device=x.device, dtype=torch.float64), inv)
    c, s = f.cos()[:, None], f.sin()[:, None]
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _conv64(x, w):
    """x (N, C, D), w (D, K): taps end at the current row, zeros before the chunk."""
    K, C = w.shape[1], x.shape[1]
    y = torch.zeros_like(x)
    for j in range(K):
        back = K - 1 - j
        if back < C:
            y[:, back:] += x[:, :C - back] * w[:, j]
    return y


def _mlp64(x, gate_up, down):
    gu = x @ gate_up.T
    I = gu.shape[-1] // 2
    return (F.silu(gu[..., :I]) * gu[..., I:]) @ down.T


def _ttt64(x, t, w, chunk, every, lr=0.3):
    """The TTT MLP: chunk c is answered with the weights that the chunks before it
    have moved; `every` chunks to a group."""
    B, T, H = x.shape
    I = w["down"].shape[1]
    n = -(-T // chunk)
    x, t = (F.pad(v, (0, 0, 0, n * chunk - T)) for v in (x, t))

    def features(v):
        gu = v @ w["gate_up"].T
        return F.silu(gu[..., :I]) * gu[..., I:]

    W_upd = w["down"].T @ w["ttt_proj"]
    out = torch.empty(B, n * chunk, H, dtype=torch.float64, device=x.device)
    every = max(1, min(n, every))
    for b in range(B):
        total, z_hat, z_tgt = torch.zeros_like(w["down"]), None, None
        for c in range(n):
            rows = slice(c * chunk, (c + 1) * chunk)
            z = features(x[b, rows])
            out[b, rows] = z @ (w["down"] + lr * total).T
            if c < n - 1:
                z_hat = _conv64(features(t[b, rows])[None], w["conv_s"][:, 0])[0]
                z_tgt = _conv64(z[None], w["conv_t"][:, 0])[0]
                beta = (t[b, rows] @ w["b_proj"]).sigmoid()
                total = total + (((z_tgt - z_hat) @ W_upd) * beta[:, None]).T @ z_hat
    return out[:, :T]


def _prefill64(case, seed):
    cfg = ipttcdv9.resolve_config(_model_cfg(case))
    w = {n: v for n, v in ipttcdv9.init_weights(cfg, torch.device(DEV, 0), seed=seed).items()}
    g = _gen(seed)
    ids = torch.randint(0, cfg["vocab_size"], (case["B"], case["T"]), generator=g, device=DEV)
    Hq, Hkv, D, C, eps = (cfg[n] for n in ("num_heads", "num_kv_heads", "head_dim", "ttt_chunk",
                                           "norm_eps"))
    kv, outs, step = {}, [], case["chunk"] or case["T"]
    for a in range(0, case["T"], step):
        part = ids[:, a:a + step]
        B, T = part.shape
        h = w["model.embeddings.weight"][part].double()
        for i in range(case["layers"]):
            p = {n[len(f"model.layers.{i}."):]: v.double() for n, v in w.items()
                 if n.startswith(f"model.layers.{i}.")}
            x = _norm64(h, p["attn_norm.weight"], eps)
            q, k, v = ((x @ p[f"attn.{n}_proj.weight"].T).view(B, T, -1, D) for n in "qkv")
            q = _rope64(_norm64(q, p["attn.q_norm.weight"], 1e-5), a)
            k = _rope64(_norm64(k, p["attn.k_norm.weight"], 1e-5), a)
            if i in kv:
                k, v = torch.cat([kv[i][0], k], 1), torch.cat([kv[i][1], v], 1)
            kv[i] = (k, v)
            is_ttt = i == 0 and T >= C
            windows = [cfg["window_size"], C * cfg["ttt_visible_chunks"]][:2 if is_ttt else 1]
            o = [_attention64(q[b], k[b], v[b], windows) for b in range(B)]
            r = [h + torch.stack([x[m][0].reshape(T, Hq * D) for x in o]) @ p["attn.o_proj.weight"].T
                 for m in range(len(windows))]
            h = r[0]
            x = [_norm64(y, p["mlp_norm.weight"], eps) for y in r]
            gate_up = torch.cat([p["mlp.gate_proj.weight"], p["mlp.up_proj.weight"]])
            if is_ttt:
                tw = dict(gate_up=gate_up, down=p["mlp.down_proj.weight"],
                          ttt_proj=p["mlp.ttt_proj.weight"], conv_t=p["mlp.ttt_teacher_conv.weight"],
                          conv_s=p["mlp.ttt_student_conv.weight"], b_proj=p["mlp.b_proj"])
                h = h + _ttt64(x[0], x[1], tw, C, cfg["ttt_update_every"])
            else:
                h = h + _mlp64(x[0], gate_up, p["mlp.down_proj.weight"])
        x = _norm64(h[:, -case["keep"]:], w["model.norm.weight"].double(), eps)
        outs.append(x @ w["lm_head.weight"].double().T)
    return outs if case["chunk"] else outs[0]


@torch.inference_mode()
def exact(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind in ("dual", "window", "lse"):
        if work(case)["flops"] > 1e13:
            return None
        q, k, v = _qkv(case, g)
        windows = [case["wt"]] if kind == "window" else [case["wt"], case["ws"]]
        each = [_attention64(q[b], k[b], v[b], windows) for b in range(case["B"])]
        got = [torch.stack([e[m][0] for e in each]) for m in range(len(windows))]
        if case["lse"]:
            got += [torch.stack([e[m][1] for e in each]) for m in range(len(windows))]
        return got if len(got) > 1 else got[0]
    if kind == "varlen":
        q, k, v = _packed(case, g)
        parts, at = [], 0
        for n in _lengths(case):
            if n:
                s = slice(at, at + n)
                parts.append(_attention64(q[s], k[s], v[s], [case["wt"], case["ws"]]))
            at += n
        got = [torch.cat([p[m][0] for p in parts]) for m in range(2)]
        if case["lse"]:
            got += [torch.cat([p[m][1] for p in parts], -1) for m in range(2)]
        return got
    if kind == "conv":
        x, w = _conv(case, g)
        return _conv64(x.double(), w.double())
    if kind == "prologue":
        q, k, w = _prologue(case, g)
        got = []
        for i, x in enumerate((q, k)):
            x = x.double()
            x = x if w is None else _norm64(x, w[i].double(), 1e-6)
            got.append(_rope64(x, case["offset"]))
        return got
    if kind == "epilogue":
        both, res, w, nw = (x.double() for x in _epilogue(case, g))
        x = [both[m] @ w.T + res for m in range(2)]
        return [_norm64(x[0], nw, 1e-6), x[0], _norm64(x[1], nw, 1e-6)]
    if kind == "ttt":
        both, w = _ttt(case, g)
        return _ttt64(both[0].double(), both[1].double(), {n: v.double() for n, v in w.items()},
                      case["chunk"], case["every"])
    return _prefill64(case, seed)
