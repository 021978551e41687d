"""The C++ autograd functions of plain eager training calls (ops.eager_ext):
when they stand aside (CPU), and that they do what the custom ops do (GPU):
the same kernels, so bit-identical outputs and gradients, and the same
behaviour with saved-tensor hooks, checkpointing, create_graph, batched
gradients, in-place changes, other streams and the backward switch.
"""
from __future__ import annotations

import pytest
import torch
from torch.autograd import forward_ad
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode
from torch.utils.checkpoint import checkpoint

import hlm_attn
from hlm_attn import ops
from oracle import linear_ce as ce_oracle


class Record(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def test_stands_aside_where_the_op_must_be_seen():
    t = torch.ones(2)
    ext = ops.eager_ext(t, torch.nn.Parameter(t))
    assert ext is not None, "the torch extension is part of the build"
    with Record():
        assert ops.eager_ext(t) is None
    with torch.device("cpu"):
        assert ops.eager_ext(t) is None  # a function mode
    with forward_ad.dual_level():
        assert ops.eager_ext(t) is None
    seen = []
    torch.func.vmap(lambda x: (seen.append(ops.eager_ext(x)), x)[1])(t)
    torch.func.grad(lambda x: (seen.append(ops.eager_ext(x)), x.sum())[1])(t)
    torch.jit.trace(lambda x: (seen.append(ops.eager_ext(x)), x + 1)[1], (t,), check_trace=False)
    assert seen and all(s is None for s in seen)

    class Sub(torch.Tensor):
        pass

    assert ops.eager_ext(t.as_subclass(Sub)) is None
    # CPU tensors and layouts of the general path are left to it
    q = torch.ones(1, 4, 2, 64, dtype=torch.bfloat16)
    assert ext.attn_train(q, q, q, 0, 0.125) is None
    assert ext.qk_norm_rope_train(q, q, t, t, 1e-6) is None
    assert ext.residual_rms_norm_train(q, q, 1e-6) is None


DEV = "cuda"


def _attn_inputs(D=64, Hkv=2, T=200):
    g = torch.Generator().manual_seed(5)
    q, k, do = (torch.randn(2, T, h, D, generator=g).bfloat16().to(DEV) for h in (4, Hkv, 4))
    fused = torch.randn(2, T, 3 * Hkv * D, generator=g).bfloat16().to(DEV)
    v = fused[..., Hkv * D : 2 * Hkv * D].view(2, T, Hkv, D)
    return [t.detach().requires_grad_(True) for t in (q, k, v)], do


def _producer_inputs():
    g = torch.Generator().manual_seed(6)
    fused = torch.randn(2, 50, 5 * 64, generator=g).bfloat16().to(DEV)
    q, k, _ = (t.view(2, 50, -1, 64) for t in fused.split((3 * 64, 64, 64), dim=-1))
    cos, sin = (torch.randn(1, 50, 1, 16, generator=g).bfloat16().to(DEV) for _ in range(2))
    return [t.detach().requires_grad_(True) for t in (q, k)], cos, sin


def _residual_inputs():
    g = torch.Generator().manual_seed(7)
    return [torch.randn(3, 37, 520, generator=g).bfloat16().to(DEV).requires_grad_(True) for _ in range(2)]


def _attention(D=64, window=70, dout=None):
    ins, do = _attn_inputs(D)
    o = hlm_attn.attention(*ins, window)
    return (o, *torch.autograd.grad(o, ins, do if dout is None else dout(do)))


def _producer():
    ins, cos, sin = _producer_inputs()
    out = hlm_attn.qk_norm_rope_hip(*ins, cos, sin, 1e-6)
    return (*out, *torch.autograd.grad(out, ins, [torch.ones_like(t) * 0.3 for t in out]))


def _producer_one_output():
    ins, cos, sin = _producer_inputs()
    out = hlm_attn.qk_norm_rope_hip(*ins, cos.float(), sin.float(), 1e-6)
    return torch.autograd.grad(out[0].float().square().sum(), ins)


def _residual():
    ins = _residual_inputs()
    out = hlm_attn.residual_rms_norm_hip(*ins, 1e-6)
    return (*out, *torch.autograd.grad((out[0].float() + 2 * out[1].float()).sum(), ins))


def _parameters():
    ins, do = _attn_inputs()
    ins = [torch.nn.Parameter(t.detach().contiguous()) for t in ins]
    hlm_attn.attention(*ins, None).backward(do)
    return [t.grad for t in ins]


def _offloaded():
    ins, do = _attn_inputs()
    with torch.autograd.graph.save_on_cpu():
        o = hlm_attn.attention(*ins, 33)
    return torch.autograd.grad(o, ins, do)


def _checkpointed():
    ins, do = _attn_inputs()
    r = _residual_inputs()
    o = checkpoint(lambda q, k, v: hlm_attn.attention(q, k, v, 64), *ins, use_reentrant=False)
    n = checkpoint(lambda a, b: hlm_attn.residual_rms_norm_hip(a, b, 1e-6)[1], *r, use_reentrant=False)
    return (*torch.autograd.grad(o, ins, do), *torch.autograd.grad(n.float().square().sum(), r))


def _retained():
    ins, do = _attn_inputs(Hkv=1, T=300)
    o = hlm_attn.attention(*ins, None)
    first = torch.autograd.grad(o, ins, do, retain_graph=True)
    return (*first, *torch.autograd.grad(o, ins, 2 * do))


def _batched_gradient():
    ins, do = _attn_inputs()
    o = hlm_attn.attention(*ins, 50)
    return torch.autograd.grad(o, ins, torch.stack((do, -do)), is_grads_batched=True)


def _side_stream():
    ins, do = _attn_inputs()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        o = hlm_attn.attention(*ins, 50)
        g = torch.autograd.grad(o, ins, do)
    torch.cuda.current_stream().wait_stream(side)
    for t in (o, *g):
        t.record_stream(torch.cuda.current_stream())
    return (o, *g)


def _chunked_inputs(D, T=1500):
    """One sequence, full causal: dQ and dK/dV both run in chunks."""
    g = torch.Generator().manual_seed(8)
    ins = [torch.randn(1, T, h, D, generator=g).bfloat16().to(DEV).requires_grad_(True) for h in (4, 2, 2)]
    assert ops.bwd_split_bytes(1, T, 4, 2, D, 0) > 0
    return ins, torch.randn(1, T, 4, D, generator=g).bfloat16().to(DEV)


def _chunked(D):
    ins, do = _chunked_inputs(D)
    o = hlm_attn.attention(*ins, None)
    return (o, *torch.autograd.grad(o, ins, do))


def _chunked_side_stream():
    """The workspace is allocated and used on the backward's stream, with work
    of another size on the main one meanwhile."""
    ins, do = _chunked_inputs(64)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        o = hlm_attn.attention(*ins, None)
        g = torch.autograd.grad(o, ins, do)
    other = _chunked(128)
    torch.cuda.current_stream().wait_stream(side)
    for t in (o, *g):
        t.record_stream(torch.cuda.current_stream())
    return (o, *g, *other)


def _lm_head(vocab):
    """2500 tokens in chunks of 2048 and 452, ignored targets, against the float64
    loss of the same bf16 values.  Roundings to bf16 (2^-9 of the value): of the
    logits (below 4, so 2^-7 of a probability at most, 1e-3 of the loss), of
    their gradient and of each product, twice for dW."""
    g = torch.Generator().manual_seed(vocab)
    hidden = torch.randn(2500, 128, generator=g).bfloat16()
    weight = (torch.randn(vocab, 128, generator=g) * 0.05).bfloat16()
    targets = torch.randint(0, vocab, (2500,), generator=g)
    targets[::7] = -100
    h, w = (t.to(DEV).requires_grad_(True) for t in (hidden, weight))
    loss = hlm_attn.fused_linear_cross_entropy_with_weight(h, w, None, targets.to(DEV), chunk_size=2048)
    grads = torch.autograd.grad(loss, (h, w))
    ref_loss, *ref, _ = ce_oracle.fused_linear_cross_entropy(hidden, weight, None, targets, 2500)
    assert abs(loss.item() - ref_loss.item()) <= 1e-3 * ref_loss.item()
    for got, want in zip(grads, ref):
        assert ((got.double().cpu() - want).norm() / want.norm()).item() <= 1e-2
    return (loss.detach(), *grads)


WAYS = {
    "attention": _attention,
    "attention_128": lambda: _attention(128, None),
    "expanded_gradient": lambda: _attention(dout=lambda do: torch.ones((), device=DEV, dtype=torch.bfloat16).expand_as(do)),
    "strided_gradient": lambda: _attention(dout=lambda do: do.transpose(1, 2).contiguous().transpose(1, 2)),
    "producer": _producer,
    "producer_one_output": _producer_one_output,
    "residual": _residual,
    "parameters": _parameters,
    "offloaded": _offloaded,
    "checkpointed": _checkpointed,
    "retained": _retained,
    "batched_gradient": _batched_gradient,
    "side_stream": _side_stream,
    "chunked": lambda: _chunked(64),
    "chunked_128": lambda: _chunked(128),
    "chunked_side_stream": _chunked_side_stream,
    "lm_head_odd": lambda: _lm_head(2049),       # rows padded to 2112 columns
    "lm_head_4_kb_rows": lambda: _lm_head(2048), # 64 columns more
    "lm_head_split": lambda: _lm_head(4097),     # dhidden with the vocabulary split
}


@pytest.mark.gpu
@pytest.mark.parametrize("way", WAYS)
def test_equals_the_custom_ops(way, monkeypatch):
    used = []
    real = ops.eager_ext
    monkeypatch.setattr(ops, "eager_ext", lambda *a: (used.append(real(*a)), used[-1])[1])
    fast = WAYS[way]()
    assert used and all(u is not None for u in used)
    monkeypatch.setattr(ops, "eager_ext", lambda *a: None)
    slow = WAYS[way]()
    torch.cuda.synchronize()
    for a, b in zip(fast, slow):
        assert a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("path", ["eager", "op"])
def test_second_derivatives_and_in_place_changes_are_refused(path, monkeypatch):
    if path == "op":
        monkeypatch.setattr(ops, "eager_ext", lambda *a: None)
    ins, do = _attn_inputs()
    o = hlm_attn.attention(*ins, 50)
    g = torch.autograd.grad(o, ins, do, create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(g[0].float().sum(), ins[0])
    r = _residual_inputs()
    out = hlm_attn.residual_rms_norm_hip(*r, 1e-6)
    g = torch.autograd.grad(out[1].float().square().sum(), r, create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(g[0].float().sum(), r[0])
    ins, do = _attn_inputs()
    q = ins[0] * 1
    o = hlm_attn.attention(q, *ins[1:], 50)
    q.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        o.backward(do)
    o = hlm_attn.attention(*ins, 50)
    o.backward(do)
    with pytest.raises(RuntimeError, match="second time"):
        o.backward(do)


@pytest.mark.gpu
def test_a_backward_under_a_dispatch_mode_shows_the_op(monkeypatch):
    ins, do = _attn_inputs()
    o = hlm_attn.attention(*ins, 50)
    plain = torch.autograd.grad(o, ins, do, retain_graph=True)
    with Record() as rec:
        seen = torch.autograd.grad(o, ins, do, retain_graph=True)
    assert any("hip_attn_bwd" in n for n in rec.names)
    assert all(torch.equal(a, b) for a, b in zip(plain, seen))
    with Record() as rec:
        hlm_attn.attention(*ins, 50)
    assert any("hip_attn_fwd" in n for n in rec.names)
    # the backward switch reaches the single-pass kernels through the op
    monkeypatch.setenv("HLM_ATTN_BWD", "fused")
    fused = torch.autograd.grad(o, ins, do)
    assert torch.equal(fused[1], plain[1]) and torch.equal(fused[2], plain[2])
    assert ((fused[0].float() - plain[0].float()).norm() / plain[0].float().norm()).item() <= 1e-2


class RecordFunctions(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


@pytest.mark.gpu
def test_a_backward_under_a_function_mode_shows_the_op():
    """torch.autograd.backward, which no function mode takes over, with the mode
    active around it only."""
    for make, name in ((_attn_inputs, "hip_attn_bwd"), (_producer_inputs, "hip_qk_norm_rope_backward"),
                       (_residual_inputs, "hip_residual_rms_norm_backward")):
        if make is _attn_inputs:
            ins, do = make()
            out, grads = [hlm_attn.attention(*ins, 50)], [do]
        elif make is _producer_inputs:
            ins, cos, sin = make()
            out = hlm_attn.qk_norm_rope_hip(*ins, cos, sin, 1e-6)
            grads = [t.detach() for t in out]
        else:
            ins = make()
            out = hlm_attn.residual_rms_norm_hip(*ins, 1e-6)
            grads = [t.detach() for t in out]
        plain = torch.autograd.grad(out, ins, grads, retain_graph=True)
        with RecordFunctions() as rec:
            torch.autograd.backward(out, grads, retain_graph=True)
        assert any(name in n for n in rec.names), rec.names
        assert all(torch.equal(a, t.grad) for a, t in zip(plain, ins))
    # an error inside the op arrives as it was raised
    ins, do = _attn_inputs()
    o = hlm_attn.attention(*ins, 50)
    bad = torch.empty(do.numel() + 1, dtype=do.dtype, device=DEV)[1:].view(do.shape)
    with RecordFunctions(), pytest.raises(RuntimeError, match="16-byte aligned"):
        torch.autograd.backward([o], [bad])


@pytest.mark.gpu
def test_inputs_of_the_general_path_still_take_it():
    """fp32 inputs run, misaligned ones and mismatched shapes are refused, as by
    the custom op."""
    ins, do = _attn_inputs()
    f32 = [t.detach().float().requires_grad_(True) for t in ins]
    o = hlm_attn.attention(*f32, 50)
    ref = hlm_attn.attention(*[t.detach() for t in ins], 50)
    assert torch.equal(o, ref) and all(g.dtype == torch.float32 for g in torch.autograd.grad(o, f32, do))
    buf = torch.empty(ins[0].numel() + 1, dtype=torch.bfloat16, device=DEV)
    q = buf[1:].view(ins[0].shape).copy_(ins[0].detach()).detach().requires_grad_(True)
    with pytest.raises(RuntimeError, match="16-byte aligned"):
        hlm_attn.attention(q, ins[1], ins[2], 50)
    with pytest.raises(RuntimeError, match="16-byte aligned"):
        torch.autograd.grad(hlm_attn.attention(*ins, 50), ins, q.detach())
    with pytest.raises(RuntimeError, match="disagree"):
        hlm_attn.attention(ins[0][:, :100], ins[1], ins[2])
    with pytest.raises(RuntimeError, match="differ"):
        a, b = _residual_inputs()
        hlm_attn.residual_rms_norm_hip(a, b[:2], 1e-6)
