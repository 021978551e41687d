"""Performance cases: the work a hackable-lm user has this library do, through its public entry points.

A model calls attention() once per layer (forward and backward in training, no-grad forwards in evaluation and
in the generation loop, which has no KV cache and runs the whole prefix again for each token), qk_norm_rope_hip()
before it, residual_rms_norm_hip() after each branch and fused_linear_cross_entropy_with_weight() once per step.
Shapes come from the configurations that bench.py and the GPU tests use, with ragged variants of them.  As in the
model, v is a strided view of the fused q/k/v projection, q and k are RMS-normalised rows, and everything is bf16.
"""
import math
import os
import sys

import torch

if os.path.abspath("hackable-lm_amd") not in sys.path:
    sys.path.insert(0, os.path.abspath("hackable-lm_amd"))

import hlm_attn  # noqa: E402

_BF16 = torch.bfloat16
_EPS = 1e-6


def _attn(name, kind, B, T, H, Hkv, D, window):
    """kind: attn_train (forward + backward) or attn_eval (no-grad forward); window 0 is plain causal."""
    return {"name": name, "kind": kind, "B": B, "T": T, "H": H, "Hkv": Hkv, "D": D, "window": window}


def listed():
    return [
        # One step of greedy generation early in a sequence: a short odd prefix at batch 1, where latency counts.
        _attn("generate_short", "attn_eval", 1, 77, 12, 12, 64, 512),
        # A full-causal layer of a long evaluation sequence at batch 1: few query tiles, long rows.
        _attn("eval_full_long", "attn_eval", 1, 2047, 12, 12, 64, 0),
        # A training micro-batch of a small model: one ragged sequence, local window.
        _attn("train_micro", "attn_train", 1, 1000, 6, 6, 64, 300),
        # A local layer of the headline training step.
        _attn("train_local", "attn_train", 8, 2048, 12, 12, 64, 512),
        # A full-causal layer of the same step.
        _attn("train_full", "attn_train", 8, 2048, 12, 12, 64, 0),
        # A local layer of the deep model with head dim 128.
        _attn("train_d128", "attn_train", 4, 4096, 12, 12, 128, 1024),
        # A long-context local layer: one sequence of 16384 tokens.
        _attn("train_long", "attn_train", 1, 16384, 16, 16, 128, 2048),
        # Grouped-query attention on ragged sequences, full causal.
        _attn("train_gqa", "attn_train", 2, 1777, 12, 4, 128, 0),
        # The q/k RMSNorm + rotary producer of the headline step, forward and backward.
        {"name": "producer", "kind": "producer", "B": 8, "T": 2048, "H": 12, "Hkv": 12, "D": 64, "R": 16},
        # Residual add + RMSNorm of the headline step's tokens, forward and backward.
        {"name": "residual_norm", "kind": "residual", "rows": 16384, "n": 768},
        # The LM head and its loss over the headline step's tokens, the default loss chunk of 4096 rows.
        {"name": "lm_head", "kind": "lm_head", "tokens": 16384, "n": 768, "V": 32768, "chunk": 4096, "ignored": 0.0},
        # The same with an odd vocabulary, a ragged token count and some ignored targets (padded batches).
        {"name": "lm_head_odd", "kind": "lm_head", "tokens": 5000, "n": 768, "V": 50257, "chunk": 4096, "ignored": 0.1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _attn_draw(rng):
    train = rng.random() < 0.6
    D = rng.choice((64, 64, 128))
    H = rng.choice((4, 6, 8, 12, 16))
    Hkv = H if rng.random() < 0.75 else rng.choice([g for g in (1, 2, 4) if H % g == 0])
    T = _log(rng, 64, 8192) if train else _log(rng, 16, 4096)
    B = _log(rng, 1, max(1, min(16, 16384 // T)))
    window = rng.choice((0, 0, rng.randrange(128, 513), 512, rng.randrange(513, 2049)))
    return _attn("", "attn_train" if train else "attn_eval", B, T, H, Hkv, D, 0 if window >= T else window)


def draw(rng):
    most = work(next(c for c in listed() if c["name"] == "train_long"))
    pick = rng.random()
    if pick < 0.7:
        case = _attn_draw(rng)
        while work(case)["flops"] > most["flops"] or work(case)["bytes"] > most["bytes"]:
            case = _attn_draw(rng)
    elif pick < 0.8:
        D = rng.choice((64, 128))
        T = _log(rng, 16, 4096)
        H = rng.choice((6, 8, 12, 16))
        case = {"kind": "producer", "B": _log(rng, 1, max(1, min(16, 16384 // T))), "T": T, "H": H, "Hkv": rng.choice((H, H, 2)), "D": D, "R": D // 4}
    elif pick < 0.9:
        case = {"kind": "residual", "rows": _log(rng, 16, 16384), "n": 64 * rng.randrange(4, 33)}
    else:
        V = rng.choice((32768, 50257, _log(rng, 1000, 65536)))
        case = {"kind": "lm_head", "tokens": _log(rng, 256, 8192), "n": 64 * rng.randrange(4, 17), "V": V, "chunk": rng.choice((2048, 4096)), "ignored": rng.choice((0.0, 0.1))}
    case.pop("name", None)
    return case


def _rms_rows(x):
    return (x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + _EPS)).to(_BF16)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*shape):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)

    kind = case["kind"]
    s = {"case": case}
    if kind in ("attn_train", "attn_eval"):
        B, T, H, Hkv, D = (case[x] for x in ("B", "T", "H", "Hkv", "D"))
        s["q"], s["k"] = _rms_rows(randn(B, T, H, D)), _rms_rows(randn(B, T, Hkv, D))
        fused = torch.empty(B, T, (H + 2 * Hkv) * D, device="cuda", dtype=_BF16)
        fused[..., (H + Hkv) * D :] = randn(B, T, Hkv * D).to(_BF16)
        s["v"] = fused[..., (H + Hkv) * D :].view(B, T, Hkv, D)
        if kind == "attn_train":
            s["do"] = randn(B, T, H, D).to(_BF16)
            for x in ("q", "k", "v"):
                s[x] = s[x].detach().requires_grad_(True)
    elif kind == "producer":
        B, T, H, Hkv, D, R = (case[x] for x in ("B", "T", "H", "Hkv", "D", "R"))
        fused = randn(B, T, (H + 2 * Hkv) * D).to(_BF16)
        q, k, _ = fused.split((H * D, Hkv * D, Hkv * D), dim=-1)
        s["q"], s["k"] = (x.view(B, T, -1, D).detach().requires_grad_(True) for x in (q, k))
        freq = 1_000_000.0 ** (-torch.arange(0, R, 2, device="cuda").float() / R)
        angles = torch.outer(torch.arange(T, device="cuda").float(), freq).repeat(1, 2)[None, :, None]
        s["cos"], s["sin"] = angles.cos().to(_BF16), angles.sin().to(_BF16)
        s["gq"], s["gk"] = randn(B, T, H, D).to(_BF16), randn(B, T, Hkv, D).to(_BF16)
    elif kind == "residual":
        for x in ("a", "b", "ga", "gn"):
            s[x] = randn(case["rows"], case["n"]).to(_BF16)
        s["a"].requires_grad_(True)
        s["b"].requires_grad_(True)
    else:
        n, V, tokens = case["n"], case["V"], case["tokens"]
        s["hidden"] = _rms_rows(randn(tokens, n)).requires_grad_(True)
        s["weight"] = (randn(V, n) * 0.02).to(_BF16).requires_grad_(True)
        t = torch.randint(0, V, (tokens,), generator=g, device="cuda")
        drop = torch.rand(tokens, generator=g, device="cuda") < case["ignored"]
        s["targets"] = torch.where(drop, torch.full_like(t, -100), t)
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "attn_eval":
        with torch.no_grad():
            return hlm_attn.attention(state["q"], state["k"], state["v"], case["window"] or None)
    if kind == "attn_train":
        ins = (state["q"], state["k"], state["v"])
        o = hlm_attn.attention(*ins, case["window"] or None)
        return (o.detach(), *torch.autograd.grad(o, ins, state["do"]))
    if kind == "producer":
        q, k = hlm_attn.qk_norm_rope_hip(state["q"], state["k"], state["cos"], state["sin"], _EPS)
        grads = torch.autograd.grad((q, k), (state["q"], state["k"]), (state["gq"], state["gk"]))
        return (q.detach(), k.detach(), *grads)
    if kind == "residual":
        out, normed = hlm_attn.residual_rms_norm_hip(state["a"], state["b"], _EPS)
        grads = torch.autograd.grad((out, normed), (state["a"], state["b"]), (state["ga"], state["gn"]))
        return (out.detach(), normed.detach(), *grads)
    loss = hlm_attn.fused_linear_cross_entropy_with_weight(
        state["hidden"], state["weight"], None, state["targets"], chunk_size=case["chunk"]
    )
    return (loss.detach(), *torch.autograd.grad(loss, (state["hidden"], state["weight"])))


def work(case):
    """Bytes: each input once, each output once.  Attention counts the unmasked (query, key) pairs, 4 D operations
    each in the forward and 12 D in a training pass (the recomputed scores are not counted)."""
    kind = case["kind"]
    if kind in ("attn_train", "attn_eval"):
        B, T, H, Hkv, D = (case[x] for x in ("B", "T", "H", "Hkv", "D"))
        W = min(case["window"] or T, T)
        pairs = W * (W + 1) // 2 + (T - W) * W
        mult, tensors = (12, 4) if kind == "attn_train" else (4, 2)
        return {"bytes": 2 * tensors * B * T * (H + Hkv) * D, "flops": mult * D * pairs * B * H}
    if kind == "producer":
        rows = case["B"] * case["T"] * (case["H"] + case["Hkv"])
        return {"bytes": 2 * 4 * rows * case["D"] + 4 * case["T"] * case["R"], "flops": 30 * rows * case["D"]}
    if kind == "residual":
        # residual, branch, both upstream gradients in; out, normed and the shared input gradient out
        return {"bytes": 2 * 7 * case["rows"] * case["n"], "flops": 16 * case["rows"] * case["n"]}
    n, V, tokens = case["n"], case["V"], case["tokens"]
    return {"bytes": 2 * 2 * n * (tokens + V) + 8 * tokens, "flops": 6 * tokens * n * V}


def tolerance(case):
    """About four times the distance of the present results from the 64-bit ones."""
    return {
        "attn_eval": {"rel": 1e-2, "max": 5e-2},
        "attn_train": {"rel": 1.2e-2, "max": 2e-1},
        "producer": {"rel": 7e-3, "max": 3e-2},
        "residual": {"rel": 7e-3, "max": 3e-2},
        "lm_head": {"rel": 1e-2, "max": 2e-1},
    }[case["kind"]]


def _attn_exact(case, s):
    B, T, H, Hkv, D = (case[x] for x in ("B", "T", "H", "Hkv", "D"))
    W = min(case["window"] or T, T)
    scale, block = 1.0 / math.sqrt(D), 512
    train = case["kind"] == "attn_train"
    outs = [[], [], [], []]
    for b in range(B):
        q = s["q"][b].detach().double().transpose(0, 1).contiguous()
        k, v = (s[x][b].detach().double().transpose(0, 1).repeat_interleave(H // Hkv, dim=0) for x in ("k", "v"))
        o, dq, dk, dv = (torch.zeros_like(q) for _ in range(4))
        do = s["do"][b].double().transpose(0, 1).contiguous() if train else None
        for q0 in range(0, T, block):
            q1, k0 = min(q0 + block, T), max(0, q0 - W + 1)
            qb, kb, vb = q[:, q0:q1].contiguous(), k[:, k0:q1].contiguous(), v[:, k0:q1].contiguous()
            lag = torch.arange(q0, q1, device=q.device)[:, None] - torch.arange(k0, q1, device=q.device)[None]
            sc = torch.matmul(qb, kb.transpose(1, 2).contiguous()) * scale
            p = torch.softmax(sc.masked_fill((lag < 0) | (lag >= W), float("-inf")), dim=-1)
            o[:, q0:q1] = torch.matmul(p, vb)
            if train:
                dob = do[:, q0:q1].contiguous()
                dp = torch.matmul(dob, vb.transpose(1, 2).contiguous())
                ds = p * (dp - (p * dp).sum(dim=-1, keepdim=True)) * scale
                dq[:, q0:q1] = torch.matmul(ds, kb)
                dk[:, k0:q1] += torch.matmul(ds.transpose(1, 2).contiguous(), qb)
                dv[:, k0:q1] += torch.matmul(p.transpose(1, 2).contiguous(), dob)
        dk, dv = (x.view(Hkv, H // Hkv, T, D).sum(dim=1) for x in (dk, dv))
        for to, x in zip(outs, (o, dq, dk, dv)):
            to.append(x.transpose(0, 1))
    stacked = [torch.stack(x) for x in outs]
    return tuple(stacked) if train else stacked[0]


def _producer_exact(case, s):
    R, res = case["R"], []
    h = R // 2
    c, sn = (s[x].double()[..., :h] for x in ("cos", "sin"))
    for x, g in (("q", "gq"), ("k", "gk")):
        x, g = s[x].detach().double(), s[g].double()
        r = torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + _EPS)
        z = x * r
        y, gz = z.clone(), g.clone()
        y[..., :h], y[..., h:R] = z[..., :h] * c - z[..., h:R] * sn, z[..., h:R] * c + z[..., :h] * sn
        gz[..., :h], gz[..., h:R] = g[..., :h] * c + g[..., h:R] * sn, g[..., h:R] * c - g[..., :h] * sn
        res.append((y, r * (gz - z * (gz * z).mean(dim=-1, keepdim=True))))
    return (res[0][0], res[1][0], res[0][1], res[1][1])


def _residual_exact(s):
    out = (s["a"].detach().float() + s["b"].detach().float()).to(_BF16).double()  # the sum is rounded by definition
    r = torch.rsqrt(out.square().mean(dim=-1, keepdim=True) + _EPS)
    z, gn = out * r, s["gn"].double()
    grad = s["ga"].double() + r * (gn - z * (gn * z).mean(dim=-1, keepdim=True))
    return (out, z, grad, grad)


def _lm_head_exact(case, s):
    hidden, weight = s["hidden"].detach().double(), s["weight"].detach().double()
    n = case["tokens"]
    loss = hidden.new_zeros(())
    dh, dw = torch.empty_like(hidden), torch.zeros_like(weight)
    w_t = weight.t().contiguous()
    for r0 in range(0, n, 1024):
        h, t = hidden[r0 : r0 + 1024], s["targets"][r0 : r0 + 1024]
        keep = t >= 0
        lp = torch.log_softmax(torch.mm(h, w_t), dim=-1)
        pick = t.clamp(min=0)[:, None]
        loss -= (lp.gather(1, pick)[:, 0] * keep).sum() / n
        g = lp.exp_()
        g.scatter_add_(1, pick, torch.full_like(pick, -1, dtype=torch.float64))
        g *= keep[:, None] / n
        dh[r0 : r0 + 1024] = torch.mm(g, weight)
        dw += torch.mm(g.t().contiguous(), h)
    return (loss, dh, dw)


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind in ("attn_train", "attn_eval"):
        return _attn_exact(case, s)
    if kind == "producer":
        return _producer_exact(case, s)
    if kind == "residual":
        return _residual_exact(s)
    return _lm_head_exact(case, s)
