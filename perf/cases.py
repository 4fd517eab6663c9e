"""The work a user of this framework has it do, as timed cases.

One BDH layer has 4 heads of N sparse neurons (x = ReLU(z), z ~ N(-1.645, 1):
about 5 % are not zero) and D value columns; the layer of the benchmark is
N = 8192, D = 256.  The paths:

  decode   one token per stream, rho [B,H,N,D] f32 updated in place
           (decode_step): what generation does for each token
  prefill  a prompt of T tokens through the RoPE-fused attention in bf16
           (try_fused_recurrent_attention_rope), from an empty or a carried
           state; with decay, the ALiBi form, whose queries carry no RoPE
           (try_fused_recurrent_attention)
  f32      the same call in f32, which an unchanged f32 model makes
  vjp      the backward of that f32 call with respect to its context
           (recurrent_attention_vjp), or of the stateless dense causal form
           (dense_causal_attention_vjp)
  layer    the whole low-rank layer around the attention, its state kept and
           continued in place (lowrank_layer_forward), T = 1 being a token
           of generation
  model    a byte-vocabulary language model of such layers, tokens to logits
           (model_forward_logits)

listed() holds one or more sizes of each path; draw() gives others of the
same ranges, ragged and odd sizes among them.
"""
import math

import numpy as np
import torch

import burn_dragon_amd as bd

HEADS = 4
THETA = 65536.0
VOCAB = 256
LAYERS = 6


def listed():
    return [
        # One user's next token: the smallest call, launches and latency.
        dict(name="decode_1", path="decode", B=1, Hv=1, T=1, N=8192, D=256, pos=1024),
        # A serving batch's next token (the decode configuration of the benchmark).
        dict(name="decode_64", path="decode", B=64, Hv=1, T=1, N=8192, D=256, pos=1024),
        # A batch of prompts (the prefill configuration of the benchmark).
        dict(name="prefill_512", path="prefill", B=8, Hv=1, T=512, N=8192, D=256, pos=0, rho=False, decay=False),
        # The next piece of two conversations: a ragged prompt onto a carried state.
        dict(name="prefill_333", path="prefill", B=2, Hv=1, T=333, N=8192, D=256, pos=777, rho=True, decay=False),
        # One long document (the long-context configuration of the benchmark).
        dict(name="prefill_8192", path="prefill", B=1, Hv=1, T=8192, N=8192, D=256, pos=0, rho=False, decay=False),
        # A small f32 model's sequence (the CPU-reference configuration of the benchmark).
        dict(name="f32_256", path="f32", B=1, Hv=1, T=256, N=1024, D=64, pos=0, rho=False, decay=False),
        # A full-size f32 batch, the forward of a training step.
        dict(name="f32_512", path="f32", B=8, Hv=1, T=512, N=8192, D=256, pos=0, rho=False, decay=False),
        # The backward of the small model, ALiBi decay, no carried state.
        dict(name="vjp_256", path="vjp", B=1, Hv=1, T=256, N=1024, D=64, rho=False, decay=True),
        # The backward of a full-size training step.
        dict(name="vjp_512", path="vjp", B=8, Hv=1, T=512, N=8192, D=256, rho=False, decay=False),
        # A ragged prompt through one layer, the state kept for generation.
        dict(name="layer_777", path="layer", B=2, T=777, N=8192, D=256, pos=0),
        # One generated token of 16 sequences through one layer.
        dict(name="layer_1", path="layer", B=16, T=1, N=8192, D=256, pos=1024),
        # Scoring a batch of texts with the 6-layer model (the model configuration of the benchmark).
        dict(name="model_1024", path="model", B=16, T=1024, N=8192, D=256, pos=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["decode", "prefill", "prefill", "f32", "vjp", "layer", "layer", "model"])
    c = dict(path=path)
    if path == "decode":
        # Any even number of neurons: RoPE turns pairs.
        c.update(B=_log(rng, 1, 64), Hv=rng.choice([1, 1, HEADS]), T=1, N=2 * _log(rng, 512, 4096),
                 D=rng.choice([64, 96, 128, 192, 256]), pos=rng.randrange(0, 65536))
    elif path == "prefill":
        B = _log(rng, 1, 8)
        c.update(B=B, Hv=rng.choice([1, 1, HEADS]), T=_log(rng, 32, 8192 // B), N=256 * _log(rng, 4, 32),
                 D=rng.choice([64, 96, 128, 192, 256]), pos=rng.randrange(0, 8192),
                 rho=rng.random() < 0.5, decay=rng.random() < 0.3)
    elif path == "f32":
        B = _log(rng, 1, 8)
        c.update(B=B, Hv=rng.choice([1, 1, HEADS]), T=_log(rng, 16, 4096 // B), N=2 * _log(rng, 256, 4096),
                 D=rng.choice([24, 64, 100, 128, 256]), pos=rng.randrange(0, 4096),
                 rho=rng.random() < 0.5, decay=rng.random() < 0.3)
    elif path == "vjp":
        B = _log(rng, 1, 8)
        c.update(B=B, Hv=rng.choice([1, 1, HEADS]), T=_log(rng, 16, 4096 // B), N=2 * _log(rng, 256, 4096),
                 D=rng.choice([24, 64, 100, 128, 256]), rho=rng.random() < 0.5, decay=rng.random() < 0.5)
    elif path == "layer":
        B = _log(rng, 1, 16)
        T = 1 if rng.random() < 0.4 else _log(rng, 2, 8192 // B)
        c.update(B=B, T=T, N=256 * _log(rng, 4, 32), D=rng.choice([64, 128, 192, 256]), pos=rng.randrange(0, 4096))
    else:
        B = _log(rng, 1, 16)
        c.update(B=B, T=_log(rng, 16, 8192 // B), N=256 * _log(rng, 4, 32), D=rng.choice([64, 128, 192, 256]), pos=0)
    return c


# ------------------------------------------------------------------ inputs --
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _sparse(g, *shape):
    return _randn(g, *shape).sub_(1.645).relu_()


def _decay():
    """The per-head ALiBi decay exp(-slope), slopes spread as a long-context model's are."""
    return torch.tensor([math.exp(-s) for s in (0.004, 0.002, 0.001, 0.0005)], device="cuda", dtype=torch.float32)


def _weights(g, N, D):
    return (_randn(g, 1, HEADS, D, N) * 0.02, _randn(g, 1, HEADS, D, N) * 0.02, _randn(g, HEADS * N, D) * 0.02)


def _inputs(case, seed):
    """The case's plain tensors."""
    g, p = _gen(seed), case["path"]
    B, T, N, D = case["B"], case["T"], case["N"], case["D"]
    if p == "decode":
        return dict(x=_sparse(g, B, HEADS, N), v=_randn(g, B, case["Hv"], D) / 16, rho=_randn(g, B, HEADS, N, D) * 0.2)
    if p in ("prefill", "f32", "vjp"):
        s = dict(x=_sparse(g, B, HEADS, T, N), v=_randn(g, B, case["Hv"], T, D) / 16)
        if p == "prefill":
            s = {k: t.to(torch.bfloat16) for k, t in s.items()}
        s["rho"] = _randn(g, B, HEADS, N, D) * 0.2 if case["rho"] else None
        s["decay"] = _decay() if case["decay"] else None
        if p == "vjp":
            s["grad"] = _randn(g, B, HEADS, T, D)
        return s
    if p == "layer":
        s = dict(weights=_weights(g, N, D), cur=torch.nn.functional.layer_norm(_randn(g, B, T, D), (D,)))
        s["rho"] = _randn(g, B, HEADS, N, D) * 0.2 if case["pos"] else torch.zeros(B, HEADS, N, D, device="cuda")
        return s
    return dict(weights=_weights(g, N, D), embed=_randn(g, VOCAB, D) * 0.02, head=_randn(g, D, VOCAB) * 0.02,
                tokens=torch.randint(0, VOCAB, (B, T), generator=g, device="cuda", dtype=torch.int32))


def prepare(case, seed):
    s = _inputs(case, seed)
    if case["path"] == "layer":
        s["weights"] = bd.LowRankWeights.pack(*s["weights"])
    elif case["path"] == "model":
        s["weights"] = bd.pack_model(s.pop("embed"), *s["weights"], s.pop("head"), LAYERS)
    s["case"] = case
    return s


# --------------------------------------------------------------------- run --
def run(state):
    c = state["case"]
    p = c["path"]
    if p == "decode":
        out = bd.decode_step(state["x"], state["v"], state["rho"], position=c["pos"])
        return {"readout": out.readout, "rho": state["rho"]}
    if p in ("prefill", "f32"):
        if c["decay"]:
            out = bd.try_fused_recurrent_attention(state["x"], state["v"], state["rho"], state["decay"])
        else:
            out = bd.try_fused_recurrent_attention_rope(state["x"], state["v"], state["rho"], position=c["pos"])
        return {"context": out.context, "rho": out.rho}
    if p == "vjp":
        if c["rho"] or not c["decay"]:
            out = bd.recurrent_attention_vjp(state["grad"], state["x"], state["v"], state["rho"], state["decay"])
            return {"query": out.grad_query, "value": out.grad_value, "rho": out.grad_rho, "decay": out.grad_decay}
        out = bd.dense_causal_attention_vjp(state["grad"], state["x"], state["v"], state["decay"])
        return {"query": out.grad_query, "value": out.grad_value, "decay": out.grad_decay}
    if p == "layer":
        out = bd.lowrank_layer_forward(state["cur"], state["weights"], position=c["pos"], rho=state["rho"],
                                       inplace=True)
        return {"next": out.next, "rho": out.rho}
    return {"logits": bd.model_forward_logits(state["tokens"], state["weights"], position=c["pos"])}


# -------------------------------------------------------------------- work --
def _attention_flops(T, N, D, state):
    """One stream: the least of the closed form over the whole sequence and
    over 128-token chunks whose state is carried."""
    whole = T * (T - 1) * (N + D) + state * 2 * T * N * D
    chunked = T * 4 * N * D + T * min(T - 1, 127) * (N + D)
    return min(whole, chunked)


def work(case):
    p, B, T, N, D = case["path"], case["B"], case["T"], case["N"], case["D"]
    S = B * HEADS
    if p == "decode":
        rows = S * N * (1 - 0.95 ** 2)  # a neuron or its RoPE partner is active
        return {"bytes": 4 * (S * N + B * case["Hv"] * D + S * D) + 8 * rows * D, "flops": 4 * rows * D}
    if p in ("prefill", "f32"):
        e = 2 if p == "prefill" else 4
        b = e * (S * T * N + B * case["Hv"] * T * D) + 4 * (S * T * D + S * N * D * (2 if case["rho"] else 1))
        f = S * (_attention_flops(T, N, D, 1) + (2 * T * N * D if case["rho"] else 0))
        return {"bytes": b, "flops": f}
    if p == "vjp":
        # S, the query's and the value's gradients, and G V^T over the triangle.
        f = S * (T * (T - 1) * (3 * N + 2 * D) + (6 * T * N * D if case["rho"] else 0))
        b = 4 * (2 * S * T * N + 2 * B * case["Hv"] * T * D + S * T * D + (2 * S * N * D if case["rho"] else 0))
        return {"bytes": b, "flops": f}
    f = 6 * B * T * HEADS * N * D
    w = 2 * 3 * HEADS * N * D
    if p == "layer":
        if T == 1:
            rows = 0.75 * S * N  # half of the neurons, and their RoPE partners
            return {"bytes": w + 8 * rows * D + 8 * B * D, "flops": f + 4 * rows * D}
        f += S * (_attention_flops(T, N, D, 1) + (2 * T * N * D if case["pos"] else 0))
        return {"bytes": w + 8 * S * N * D + 8 * B * T * D, "flops": f}
    f = LAYERS * (f + S * _attention_flops(T, N, D, 0)) + 2 * B * T * D * VOCAB
    return {"bytes": w + 4 * B * T * (1 + VOCAB) + 4 * VOCAB * D + 2 * VOCAB * D, "flops": f}


def tolerance(case):
    """About four times the path's measured error against 64 bits: 1e-6 in
    f32 (1.7e-6 for a decode step's readout, whose turns at late positions
    round to 32 bits), 2.5e-3 for one bf16 attention, 3.5e-3 for a layer of
    bf16 products, 8e-3 after six of them."""
    return {"rel": {"decode": 7e-6, "f32": 4e-6, "vjp": 4e-6, "prefill": 1e-2, "layer": 1.4e-2, "model": 3e-2}[case["path"]]}


# ------------------------------------------------------------------- exact --
def _freqs(N):
    """Turns per position of each neuron, rounded to 32 bits after each step as the model defines them."""
    i = np.arange(N)
    e = (i // 2 * 2).astype(np.float32) / np.float32(N)
    f = np.float32(1) / np.power(THETA, e.astype(np.float64)).astype(np.float32)
    return torch.from_numpy(f / (np.float32(2) * np.float32(np.pi))).cuda()


def _rope64(x, pos, freqs):
    """Rows x [T, N] in 64 bits at positions pos.., the turn p f mod 1 in 32
    bits as the model defines it."""
    p = torch.arange(pos, pos + x.shape[0], device="cuda", dtype=torch.float32)
    raw = p[:, None] * freqs[None, ::2]
    a = (raw - raw.floor()).double() * (2 * math.pi)
    c, s = a.cos(), a.sin()
    out = torch.empty_like(x)
    out[:, ::2] = x[:, ::2] * c - x[:, 1::2] * s
    out[:, 1::2] = x[:, 1::2] * c + x[:, ::2] * s
    return out


def _gap(T, d):
    """d^(r-c) below the diagonal, 0 on and above it."""
    t = torch.arange(T, device="cuda", dtype=torch.float64)
    g = (t[:, None] - t[None, :])
    return torch.where(g > 0, d ** g.clamp(min=0), torch.zeros_like(g))


def _attention64(q, v, rho, d):
    T = q.shape[0]
    ctx = (q @ q.T).mul_(_gap(T, d)) @ v
    t = torch.arange(T, device="cuda", dtype=torch.float64)[:, None]
    new = (q * d ** (T - t)).T @ v
    if rho is not None:
        ctx += (q @ rho) * d ** t
        new += d ** T * rho
    return ctx, new


def _norm64(x):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), eps=1e-5)


def _layer64(cur, weights, pos, rho, freqs):
    """One row's layer: cur [T, D], rho [H, N, D] or None -> next, rho."""
    enc, encv, dec = weights
    z, states = 0.0, []
    N = enc.shape[-1]
    for h in range(HEADS):
        x = (cur @ enc[0, h].double()).relu_()
        a, r = _attention64(_rope64(x, pos, freqs), cur, rho[h].double() if rho is not None else None, 1.0)
        y = (_norm64(a) @ encv[0, h].double()).relu_().mul_(x)
        z = z + y @ dec[h * N:(h + 1) * N].double()
        states.append(r)
    return _norm64(cur + _norm64(z)), torch.stack(states)


def _vjp64(q, v, g, rho, d):
    T = q.shape[0]
    D = _gap(T, d)
    t = torch.arange(T, device="cuda", dtype=torch.float64)[:, None]
    S, GS = (q @ q.T) * D, g @ v.T
    W = GS * D
    gq, gv = (W + W.T) @ q, S.T @ g
    gd = (GS * S * (t - t.T).clamp(min=0)).sum() / d
    gr = None
    if rho is not None:
        gt = g * d ** t
        gq += gt @ rho.T
        gd = gd + (gt * (q @ rho) * t).sum() / d
        gr = q.T @ gt
    return gq, gv, gd, gr


def exact(case, seed):
    s, p = _inputs(case, seed), case["path"]
    B, T, N, D = case["B"], case["T"], case["N"], case["D"]
    freqs = _freqs(N)
    if p == "decode":
        outs, rho = [], s["rho"].double()
        for b in range(B):
            for h in range(HEADS):
                q = _rope64(s["x"][b, h].double()[None], case["pos"], freqs)[0]
                outs.append(q @ rho[b, h])
                rho[b, h].addr_(q, s["v"][b, h % case["Hv"]].double())
        return {"readout": torch.stack(outs).view(B, HEADS, D), "rho": rho}
    if p in ("prefill", "f32"):
        ctx, rho = torch.empty(B, HEADS, T, D, device="cuda", dtype=torch.float64), []
        for b in range(B):
            for h in range(HEADS):
                q = s["x"][b, h].double()
                d = 1.0
                if case["decay"]:
                    d = float(s["decay"][h])
                else:
                    q = _rope64(q, case["pos"], freqs)
                ctx[b, h], r = _attention64(q, s["v"][b, h % case["Hv"]].double(),
                                            s["rho"][b, h].double() if case["rho"] else None, d)
                rho.append(r)
        return {"context": ctx, "rho": torch.stack(rho).view(B, HEADS, N, D)}
    if p == "vjp":
        gq = torch.empty(B, HEADS, T, N, device="cuda", dtype=torch.float64)
        gv = torch.zeros(B, case["Hv"], T, D, device="cuda", dtype=torch.float64)
        gd = torch.zeros(HEADS, device="cuda", dtype=torch.float64)
        gr = []
        for b in range(B):
            for h in range(HEADS):
                d = float(s["decay"][h]) if case["decay"] else 1.0
                gq[b, h], v, dd, r = _vjp64(s["x"][b, h].double(), s["v"][b, h % case["Hv"]].double(),
                                            s["grad"][b, h].double(), s["rho"][b, h].double() if case["rho"] else None, d)
                gv[b, h % case["Hv"]] += v
                gd[h] += dd
                gr.append(r)
        out = {"query": gq, "value": gv, "decay": gd}
        if case["rho"] or not case["decay"]:
            out["rho"] = torch.stack(gr).view(B, HEADS, N, D) if case["rho"] else None
        return out
    if p == "layer":
        rows = [_layer64(s["cur"][b].double(), s["weights"], case["pos"], s["rho"][b], freqs) for b in range(B)]
        return {"next": torch.stack([r[0] for r in rows]), "rho": torch.stack([r[1] for r in rows])}
    logits = []
    for b in range(B):
        cur = _norm64(s["embed"].double()[s["tokens"][b].long()])
        for _ in range(LAYERS):
            cur, _rho = _layer64(cur, s["weights"], case["pos"], None, freqs)
        logits.append(cur @ s["head"].double())
    return {"logits": torch.stack(logits)}
