"""The LM-head loss's chunk loop (kernels._LMHeadLoss) on the CPU: the library
products run as on the GPU, the cross-entropy rows come from the oracle in
place of their launch.  And how torch.compile sees the loss: traced with fake
ROCm tensors."""
from __future__ import annotations

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils.flop_counter import FlopCounterMode

import hlm_attn
from hlm_attn import kernels, ops
from oracle import linear_ce as oracle


@pytest.fixture
def cpu_rows(monkeypatch):
    """linear_ce_impl without its launch: the oracle's rows, in place."""

    def rows(logits, targets, n_tokens, loss=None):
        row_loss, grad = oracle.ce_rows(logits, targets, n_tokens)
        logits.copy_(grad)
        loss = torch.empty(logits.shape[0]) if loss is None else loss
        return loss.copy_(row_loss)

    monkeypatch.setattr(ops, "linear_ce_impl", rows)


def _column_slice(t):
    wide = torch.zeros(t.shape[0], t.shape[1] + 3)
    wide[:, : t.shape[1]] = t
    return wide[:, : t.shape[1]]


LAYOUTS = {
    "contiguous": lambda t: t.clone(),
    "column_slice": _column_slice,
    "transposed": lambda t: t.t().contiguous().t(),
    "every_second_row": lambda t: t.repeat_interleave(2, dim=0)[::2],
}


@pytest.mark.parametrize("hidden_layout", LAYOUTS)
@pytest.mark.parametrize("weight_layout", LAYOUTS)
def test_every_layout_of_the_inputs_gets_its_gradients(cpu_rows, hidden_layout, weight_layout):
    """fp32: the same products of the same values, so the gradients agree with
    those of the oracle's dense form to fp32 sums (1e-5 of the largest)."""
    g = torch.Generator().manual_seed(3)
    hidden, weight, bias = (torch.randn(s, generator=g) for s in ((2500, 16), (33, 16), (33,)))
    targets = torch.randint(0, 33, (2500,), generator=g)
    targets[7] = -100
    h = LAYOUTS[hidden_layout](hidden).requires_grad_(True)
    w = LAYOUTS[weight_layout](weight).requires_grad_(True)
    b = bias.clone().requires_grad_(True)
    loss = kernels._LMHeadLoss.apply(h, w, targets, b, 2048)
    grads = torch.autograd.grad(loss, (h, w, b), allow_unused=True)
    ref_loss, *ref = oracle.fused_linear_cross_entropy(hidden, weight, bias, targets, 2500)
    assert abs(loss.item() - ref_loss.item()) <= 1e-5 * ref_loss.item()
    for name, got, want in zip(("hidden", "weight", "bias"), grads, ref):
        assert got is not None, f"{name}'s gradient is lost"
        assert (got.double() - want).abs().max().item() <= 1e-5 * want.abs().max().item(), name


@pytest.mark.parametrize("wanted", [(0,), (1,), (2,), (0, 2)])
def test_only_the_wanted_gradients_are_formed(cpu_rows, wanted):
    ins = [torch.randn(20, 8), torch.randn(5, 8), torch.randn(5)]
    for i in wanted:
        ins[i].requires_grad_(True)
    loss = kernels._LMHeadLoss.apply(ins[0], ins[1], torch.randint(0, 5, (20,)), ins[2], None)
    loss.backward()
    assert [t.grad is not None for t in ins] == [i in wanted for i in range(3)]


@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("vocab", [512, 1000, 2048, 32768, 50257, 65536])
def test_loss_traces_with_fullgraph_as_one_op(vocab, with_bias):
    """The reference trains under torch.compile(fullgraph=True)
    (kernels.py:126-137).  Vocabularies whose workspace rows are padded, for
    their alignment or off a multiple of 4 KB, and ones whose rows are not."""
    calls = []

    def backend(gm, example_inputs):
        calls.extend(str(n.target) for m in gm.modules() if isinstance(m, torch.fx.GraphModule)
                     for n in m.graph.nodes if n.op == "call_function")
        return gm.forward

    def loss_of(h, w, b, t):
        return hlm_attn.fused_linear_cross_entropy_with_weight(h, w, b, t, chunk_size=2048)

    torch._dynamo.reset()
    with FakeTensorMode(allow_non_fake_inputs=True):
        h, w, b = (torch.empty(s, dtype=torch.bfloat16, device="cuda", requires_grad=True)
                   for s in ((2500, 64), (vocab, 64), (vocab,)))
        targets = torch.empty(2500, dtype=torch.int64, device="cuda")
        loss = torch.compile(loss_of, fullgraph=True, backend=backend)(h, w, b if with_bias else None, targets)
    assert loss.shape == () and loss.dtype == torch.float32
    assert [c for c in calls if "hackable_lm" in c] == ["hackable_lm.hip_lm_head_loss.default"], calls


@pytest.mark.parametrize("grad", [True, False])
def test_a_traced_loss_forms_no_gradients_without_grad_mode(grad):
    """The op's products cannot be dropped from a graph as dead code, so a
    compiled no-grad loss (an evaluation) must not ask for them, whatever its
    inputs require."""
    flags = []

    def backend(gm, example_inputs):
        flags.extend(n.args[-3:] for m in gm.modules() if isinstance(m, torch.fx.GraphModule)
                     for n in m.graph.nodes if "hip_lm_head_loss" in str(n.target))
        return gm.forward

    torch._dynamo.reset()
    with FakeTensorMode(allow_non_fake_inputs=True), torch.set_grad_enabled(grad):
        h, w, b = (torch.empty(s, dtype=torch.bfloat16, device="cuda", requires_grad=True) for s in ((96, 64), (1000, 64), (1000,)))
        targets = torch.empty(96, dtype=torch.int64, device="cuda")
        torch.compile(hlm_attn.fused_linear_cross_entropy_with_weight, fullgraph=True, backend=backend)(h, w, b, targets)
    assert flags == [(grad, grad, grad)]


@pytest.mark.parametrize("wanted,products", [((), 1), ((0,), 2), ((0, 1, 2), 3)])
def test_the_op_and_the_direct_loop_agree(cpu_rows, wanted, products):
    """A dispatch mode sees the op, with the FLOPs of its products."""
    g = torch.Generator().manual_seed(4)
    ins = [torch.randn(s, generator=g) for s in ((2100, 8), (65, 8), (65,))]
    for i in wanted:
        ins[i].requires_grad_(True)
    targets = torch.randint(0, 65, (2100,), generator=g)

    def once():
        loss = kernels._LMHeadLoss.apply(ins[0], ins[1], targets, ins[2], 2048)
        return (loss.detach(), *(torch.autograd.grad(loss, [ins[i] for i in wanted]) if wanted else ()))

    direct = once()
    with FlopCounterMode(display=False) as flops:
        op = once()
    assert flops.get_total_flops() == products * 2 * 2100 * 65 * 8
    assert all(torch.equal(a, b) for a, b in zip(direct, op))
