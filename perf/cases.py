"""Performance cases of the framework's public entry points.

``listed()`` names the work a training or sampling program hands to this library: frozen int8
linears with LoRA adapters (``lora_forward`` / ``lora_backward``, the autograd rule, the plain
``linear``), the feed-forward block with its GELU, tiled attention forward and backward, and the
packing of weights. ``draw(rng)`` gives more cases over the same ranges of sizes, types and options.

A case is a dict of plain values; ``prepare`` makes what a program holds before the call (packed
weights, adapters, activations), ``run`` is one pass, ``exact`` the same result in 64 bits from
plain torch.
"""
from __future__ import annotations

import math

import torch

import reels_amd as ra
from reels_amd import attention as att
from reels_amd import layers

_DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_SIZE = {"bf16": 2, "f16": 2, "f32": 4}
_DEV = "cuda"


# ---- the cases -----------------------------------------------------------------------------------
def listed():
    return [
        # one conditioning vector through a frozen dense layer with bias (a time embedding's
        # projection): the smallest call, no adapter, forward only
        dict(name="dense_one_token", op="dense", M=1, K=1536, N=9216, dtype="bf16"),
        # cross-attention key / value projection of a text prompt, forward and backward
        dict(name="text_projection", op="lora", M=333, K=5120, N=5120, r=32, dtype="bf16",
             bias=False, train_bias=False, api="layer"),
        # the CPU-runnable workload's linear in the reference's own compute precision
        dict(name="short_f16", op="lora", M=1024, K=1536, N=1536, r=16, dtype="f16",
             bias=True, train_bias=False, api="layer"),
        # attention projection of the large video model at full clip length, one training step's
        # forward and backward through autograd (f32 master adapters)
        dict(name="video_projection", op="lora", M=32760, K=5120, N=5120, r=32, dtype="bf16",
             bias=False, train_bias=False, api="autograd"),
        # feed-forward block of the small video model on a six-latent-frame clip, forward and
        # backward with the GELU between the two projections and trained biases
        dict(name="feed_forward", op="ffn", M=9360, K=1536, N=8960, r=32, dtype="bf16"),
        # a projection in Float32 compute (the reference's reference precision), three latent
        # frames, forward and backward with a trained bias
        dict(name="projection_f32", op="lora", M=4680, K=1536, N=8960, r=32, dtype="f32",
             bias=True, train_bias=True, api="raw"),
        # a layer whose widths are no multiples of the tiles
        dict(name="ragged_widths", op="lora", M=777, K=1000, N=3000, r=8, dtype="bf16",
             bias=True, train_bias=False, api="layer"),
        # self-attention of the small video model at full clip length, forward and backward
        dict(name="self_attention", op="attn", B=1, Sq=32760, Sk=32760, H=12, D=128, dtype="bf16",
             causal=False, mask=False),
        # cross-attention of video tokens on a text prompt, forward and backward
        dict(name="cross_attention", op="attn", B=1, Sq=9360, Sk=512, H=40, D=128, dtype="bf16",
             causal=False, mask=False),
        # attention in Float32 compute over one latent frame, forward and backward
        dict(name="attention_f32", op="attn", B=1, Sq=1560, Sk=1560, H=12, D=128, dtype="f32",
             causal=False, mask=False),
        # attention at a head dim that is neither 64 nor 128, two sequences
        dict(name="attention_head_80", op="attn", B=2, Sq=1024, Sk=1024, H=16, D=80, dtype="bf16",
             causal=False, mask=False),
        # packing of a feed-forward weight as it is loaded
        dict(name="pack_weight", op="pack", N=13824, K=5120, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_WIDTHS = [256, 512, 768, 1024, 1536, 2048, 2560, 3072, 4096, 5120, 8960, 13824]
_RANKS = [3, 4, 8, 16, 24, 32, 64, 128]


def draw(rng):
    op = rng.choice(["dense", "lora16", "lora16", "lora32", "ragged", "ffn", "attn", "attn_any",
                     "attn_any", "pack"])
    if op == "dense":
        return dict(op="dense", M=_log(rng, 1, 77), K=rng.choice(_WIDTHS), N=rng.choice(_WIDTHS),
                    dtype=rng.choice(["bf16", "f16", "f32"]))
    if op in ("lora16", "lora32"):
        K, N = rng.choice(_WIDTHS), rng.choice(_WIDTHS)
        train = rng.random() < 0.3
        dtype = rng.choice(["bf16", "f16"]) if op == "lora16" else "f32"
        # a pass costs 4 M K N operations or so; f32 runs at a small part of the 16-bit rate
        most = min(32760, int((8e11 if dtype != "f32" else 4e10) / (K * N)))
        return dict(op="lora", M=_log(rng, 16, max(most, 64)), K=K, N=N, r=rng.choice(_RANKS),
                    dtype=dtype, bias=train or rng.random() < 0.5, train_bias=train,
                    api="raw" if train else rng.choice(["layer", "raw", "autograd"]))
    if op == "ragged":
        return dict(op="lora", M=_log(rng, 1, 1500), K=_log(rng, 100, 3000), N=_log(rng, 100, 3000),
                    r=rng.choice(_RANKS[:6]), dtype=rng.choice(["bf16", "f16", "f32"]),
                    bias=rng.random() < 0.5, train_bias=False, api="layer")
    if op == "ffn":
        K, N = rng.choice([(512, 2048), (1536, 8960), (2048, 8192), (3072, 8192)])
        return dict(op="ffn", M=_log(rng, 64, 12000), K=K, N=N, r=rng.choice(_RANKS[2:]),
                    dtype=rng.choice(["bf16", "f16"]))
    if op == "attn":
        Sq = _log(rng, 64, 16000)
        Sk = Sq if rng.random() < 0.5 else _log(rng, 16, 1024)
        return dict(op="attn", B=1 if Sq > 4000 else rng.choice([1, 2]), Sq=Sq, Sk=Sk,
                    H=rng.choice([8, 12, 16, 24, 40]), D=rng.choice([64, 128, 128]),
                    dtype=rng.choice(["bf16", "f16"]), causal=rng.random() < 0.2, mask=False)
    if op == "attn_any":
        Sq = _log(rng, 16, 2048)
        Sk = Sq if rng.random() < 0.6 else _log(rng, 16, 1024)
        f32 = rng.random() < 0.5
        opt = rng.random()
        return dict(op="attn", B=rng.choice([1, 2]), Sq=Sq, Sk=Sk, H=rng.choice([4, 8, 12, 16]),
                    D=rng.choice([32, 40, 64, 80, 96, 100, 128]) if f32
                    else rng.choice([32, 40, 72, 80, 96, 100, 112]),
                    dtype="f32" if f32 else rng.choice(["bf16", "f16"]), causal=opt < 0.2,
                    mask=0.2 <= opt < 0.4)
    return dict(op="pack", N=_log(rng, 64, 13824), K=rng.choice(_WIDTHS + [100, 1000, 1537]),
                dtype=rng.choice(["bf16", "bf16", "f16", "f32"]))


# ---- inputs --------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=_DEV).manual_seed(seed)


def _randn(g, shape, sigma, dtype):
    return (torch.randn(shape, generator=g, device=_DEV) * sigma).to(dtype)


def _codes(g, N, K):
    """Codes [N][K] and scales [N] of a weight ~N(0, 0.02), as packing gives them."""
    w = torch.randn((N, K), generator=g, device=_DEV) * 0.02
    s = w.abs().amax(dim=1) / 127.0
    return torch.round(w / s[:, None]).clamp(-127, 127).to(torch.int8), s


def _linear_inputs(case, seed):
    g = _gen(seed)
    M, K, N, r = case["M"], case["K"], case["N"], case.get("r", 0)
    dt = _DT[case["dtype"]]
    st = {}
    st["q"], st["s"] = _codes(g, N, K)
    st["x"] = _randn(g, (M, K), 1.0, dt)
    if case["op"] == "ffn":
        st["q2"], st["s2"] = _codes(g, K, N)
        st["A2"], st["B2"] = _randn(g, (N, r), 0.01, dt), _randn(g, (r, K), 0.01, dt)
        st["bias2"] = _randn(g, (K,), 0.1, dt)
        st["dy"] = _randn(g, (M, K), 1.0, dt)
    else:
        st["dy"] = _randn(g, (M, N), 1.0, dt)
    if r:
        # autograd cases keep f32 master adapters, rounded to the compute type inside the call
        ad = torch.float32 if case.get("api") == "autograd" else dt
        st["A"], st["B"] = _randn(g, (K, r), 0.01, ad), _randn(g, (r, N), 0.01, ad)
    biased = case["op"] in ("dense", "ffn") or case["bias"]
    st["bias"] = _randn(g, (N,), 0.1, dt) if biased else None
    return st


def _attention_inputs(case, seed):
    g = _gen(seed)
    B, Sq, Sk, H, D, dt = (case["B"], case["Sq"], case["Sk"], case["H"], case["D"],
                           _DT[case["dtype"]])
    st = {n: _randn(g, (B, s, H, D), 1.0, dt) for n, s in (("q", Sq), ("k", Sk), ("v", Sk),
                                                            ("dy", Sq))}
    st["mask"] = None
    if case["mask"]:  # 70% of the pairs visible; every query sees key 0
        st["mask"] = torch.rand((Sq, Sk), generator=g, device=_DEV) < 0.7
        st["mask"][:, 0] = True
    return st


def _pack_input(case, seed):
    """A frozen weight ~N(0, 0.02) with 0.1% outliers at 20 sigma."""
    g = _gen(seed)
    shape = (case["N"], case["K"])
    w = torch.randn(shape, generator=g, device=_DEV) * 0.02
    w = torch.where(torch.rand(shape, generator=g, device=_DEV) < 1e-3, w * 20.0, w)
    return w.to(_DT[case["dtype"]])


def prepare(case, seed):
    op = case["op"]
    if op == "pack":
        return dict(case=case, w=_pack_input(case, seed))
    if op == "attn":
        return dict(case=case, **_attention_inputs(case, seed))
    st = dict(case=case, **_linear_inputs(case, seed))
    dt = _DT[case["dtype"]]
    st["W"] = ra.QuantizedMatrix(st["q"], st["s"], dt)
    if op == "dense":
        st["layer"] = ra.DenseLayer(st["W"], st["bias"])
    elif op == "ffn":
        st["W2"] = ra.QuantizedMatrix(st["q2"], st["s2"], dt)
    elif case["api"] == "layer":
        st["layer"] = ra.LoRALinear(st["W"], case["r"], bias=st["bias"], A=st["A"], B=st["B"])
    elif case["api"] == "autograd":
        for n in ("x", "A", "B"):
            st[n].requires_grad_(True)
    return st


# ---- one pass ------------------------------------------------------------------------------------
def run(st):
    case = st["case"]
    op = case["op"]
    if op == "dense":
        return ra.linear(st["layer"], st["x"])
    if op == "lora":
        x, dy = st["x"], st["dy"]
        if case["api"] == "layer":
            y, h = ra.lora_forward(st["layer"], x, save_h=True)
            g = ra.lora_backward(st["layer"], x, dy, h=h)
            return y, g["dx"], g["A"], g["B"]
        if case["api"] == "autograd":
            y = layers.I8LoRALinearFunction.apply(x, st["A"], st["B"], st["q"], st["s"],
                                                  st["bias"], 1.0)
            dx, dA, dB = torch.autograd.grad(y, (x, st["A"], st["B"]), dy)
            return y.detach(), dx, dA, dB
        y, h = ra.i8lora_forward(x, st["W"], st["A"], st["B"], st["bias"], 1.0, save_h=True)
        return (y,) + tuple(ra.i8lora_backward(dy, x, st["W"], st["A"], st["B"], 1.0, h=h,
                                               want_dbias=case["train_bias"]))
    if op == "ffn":
        x, dy = st["x"], st["dy"]
        z, a, h1 = ra.i8lora_forward_gelu(x, st["W"], st["A"], st["B"], st["bias"], 1.0,
                                          save_h=True)
        y, h2 = ra.i8lora_forward(a, st["W2"], st["A2"], st["B2"], st["bias2"], 1.0, save_h=True)
        dz, dA2, dB2, db2 = ra.i8lora_backward_gelu(dy, a, z, st["W2"], st["A2"], st["B2"], 1.0,
                                                    h=h2, want_dbias=True)
        dx, dA, dB, db = ra.i8lora_backward(dz, x, st["W"], st["A"], st["B"], 1.0, h=h1,
                                            want_dbias=True)
        return y, dx, dA, dB, db, dA2, dB2, db2
    if op == "attn":
        out, cache = att.memory_efficient_attention(st["q"], st["k"], st["v"], mask=st["mask"],
                                                    causal=case["causal"])
        g = att.memory_efficient_attention_backward(st["q"], st["k"], st["v"], st["dy"], cache)
        return out, cache.logsumexp, g.q, g.k, g.v
    qm = ra.quantize_frozen_matrix(st["w"])
    return qm.values, qm.scales


# ---- the work of one pass ------------------------------------------------------------------------
def work(case):
    op = case["op"]
    e = _SIZE[case["dtype"]]
    if op == "pack":
        n = case["N"] * case["K"]
        return {"bytes": n * (e + 1) + 4 * case["N"], "flops": 3 * n}
    if op == "attn":
        B, Sq, Sk, H, D = case["B"], case["Sq"], case["Sk"], case["H"], case["D"]
        pairs = Sq * Sk
        if case["causal"]:
            m = min(Sq, Sk)
            pairs = m * (m + 1) // 2 + max(Sq - Sk, 0) * Sk
        # forward q, k, v -> out, lse; backward q, k, v, out, dy, lse -> dq, dk, dv
        size = B * H * D * e
        nbytes = size * (2 * Sq + 2 * Sk) + size * (4 * Sq + 4 * Sk) + 8 * B * H * Sq
        if case["mask"]:
            nbytes += Sq * Sk
        return {"bytes": nbytes, "flops": 14 * B * H * D * pairs}
    M, K, N = case["M"], case["K"], case["N"]
    if op == "dense":
        return {"bytes": N * K + 4 * N + e * (M * K + M * N + N), "flops": 2 * M * N * K}
    r = case["r"]
    adapters = (K + N) * r
    if op == "lora":
        # forward x, W, A, B -> y; backward dy, x, W, A, B -> dx, dA, dB
        return {"bytes": 2 * N * K + 8 * N + e * (3 * M * K + 2 * M * N + 2 * adapters)
                + 4 * adapters,
                "flops": 4 * M * N * K + 6 * M * adapters}
    # two projections; the hidden activations z, a (and dz) are written once and read in the
    # backward
    return {"bytes": 4 * N * K + 8 * (N + K) + e * (3 * M * K + 2 * M * K + 7 * M * N
                                                   + 4 * adapters) + 8 * adapters,
            "flops": 8 * M * N * K + 12 * M * adapters}


def tolerance(case):
    op, dtype = case["op"], case["dtype"]
    if op == "pack":
        return "exact"
    if op == "attn":
        return {"bf16": {"rel": 1e-2}, "f16": {"rel": 2e-3}, "f32": {"rel": 1e-5}}[dtype]
    if op == "ffn":  # a chain of four projections and a GELU
        return {"bf16": {"rel": 2e-2}, "f16": {"rel": 3e-3}}[dtype]
    return {"bf16": {"rel": 1e-2}, "f16": {"rel": 2e-3}, "f32": {"rel": 1e-5}}[dtype]


# ---- the same in 64 bits -------------------------------------------------------------------------
def _rounded(case, t):
    """An adapter as the call sees it: rounded to the compute type."""
    return t.detach().to(_DT[case["dtype"]]).double()


def _gelu64(x):
    k = math.sqrt(2.0 / math.pi)
    return 0.5 * x * (1.0 + torch.tanh(k * (x + 0.044715 * x ** 3)))


def _gelu_grad64(x):
    k = math.sqrt(2.0 / math.pi)
    t = torch.tanh(k * (x + 0.044715 * x ** 3))
    return 0.5 * (1.0 + t) + 0.5 * x * (1.0 - t * t) * k * (1.0 + 3 * 0.044715 * x * x)


def _linear64(x, W, A, B, bias):
    y = x @ W.t()
    if A is not None:
        y = y + (x @ A) @ B
    return y if bias is None else y + bias.double()


def _linear64_back(dy, x, W, A, B):
    u = dy @ B.t()
    return dy @ W + u @ A.t(), x.t() @ u, (x @ A).t() @ dy


def _attention64(case, st):
    B, Sq, Sk, H, D = case["B"], case["Sq"], case["Sk"], case["H"], case["D"]
    sc = 1.0 / math.sqrt(D)
    out, dq = (torch.empty((B, Sq, H, D), dtype=torch.float64, device=_DEV) for _ in range(2))
    dk, dv = (torch.zeros((B, Sk, H, D), dtype=torch.float64, device=_DEV) for _ in range(2))
    lse = torch.empty((B, H, Sq), dtype=torch.float64, device=_DEV)
    keys = torch.arange(Sk, device=_DEV)
    for b in range(B):
        for h in range(H):
            k, v = st["k"][b, :, h].double(), st["v"][b, :, h].double()
            for i in range(0, Sq, 4096):
                j = min(i + 4096, Sq)
                q, dy = st["q"][b, i:j, h].double(), st["dy"][b, i:j, h].double()
                s = (q @ k.t()) * sc
                if case["causal"]:
                    s.masked_fill_(keys[None, :] > torch.arange(i, j, device=_DEV)[:, None],
                                   -math.inf)
                if case["mask"]:
                    s.masked_fill_(~st["mask"][i:j], -math.inf)
                l = torch.logsumexp(s, dim=1)
                p = s.sub_(l[:, None]).exp_()
                o = p @ v
                out[b, i:j, h], lse[b, h, i:j] = o, l
                dv[b, :, h] += p.t() @ dy
                ds = p.mul_(dy @ v.t() - (dy * o).sum(dim=1, keepdim=True))
                dq[b, i:j, h] = (ds @ k) * sc
                dk[b, :, h] += (ds.t() @ q) * sc
    return out, lse, dq, dk, dv


def exact(case, seed):
    op = case["op"]
    if op == "pack":
        # quotients of two f32 values in 64 bits, rounded once more to f32: correctly rounded
        w = _pack_input(case, seed)
        top = w.float().abs().amax(dim=1).double()
        s = torch.where(top == 0, torch.ones_like(top), top / 127.0).float()
        q = torch.empty(w.shape, dtype=torch.int8, device=_DEV)
        for i in range(0, case["N"], 2048):
            t = (w[i:i + 2048].double() / s[i:i + 2048].double()[:, None]).float()
            q[i:i + 2048] = torch.round(t.clamp(-127, 127)).to(torch.int8)
        return q, s
    if op == "attn":
        return _attention64(case, _attention_inputs(case, seed))
    st = _linear_inputs(case, seed)
    W = st["q"].double() * st["s"].double()[:, None]
    x = st["x"].double()
    if op == "dense":
        return _linear64(x, W, None, None, st["bias"])
    A, B = _rounded(case, st["A"]), _rounded(case, st["B"])
    dy = st["dy"].double()
    if op == "lora":
        res = (_linear64(x, W, A, B, st["bias"]),) + _linear64_back(dy, x, W, A, B)
        return res + (dy.sum(dim=0),) if case["train_bias"] else res
    W2 = st["q2"].double() * st["s2"].double()[:, None]
    A2, B2 = _rounded(case, st["A2"]), _rounded(case, st["B2"])
    z = _linear64(x, W, A, B, st["bias"])
    a = _gelu64(z)
    y = _linear64(a, W2, A2, B2, st["bias2"])
    da, dA2, dB2 = _linear64_back(dy, a, W2, A2, B2)
    db2 = dy.sum(dim=0)
    dz = da * _gelu_grad64(z)
    dx, dA, dB = _linear64_back(dz, x, W, A, B)
    return y, dx, dA, dB, dz.sum(dim=0), dA2, dB2, db2
