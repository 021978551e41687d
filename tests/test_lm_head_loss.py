"""The LM-head loss's chunk loop (kernels._LMHeadLoss) on the CPU: the library
products run as on the GPU, the cross-entropy rows come from the oracle in
place of their launch."""
from __future__ import annotations

import pytest
import torch

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
