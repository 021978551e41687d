"""The cross-entropy rows on layouts whose rows begin or end inside a 16-byte
chunk, and at the edges of the kernel's chunk counts (GPU only).

Tolerances as in test_gpu_lm_head: loss * n within 1e-4, gradient * n within
2^-8 |ref| + 1e-6 (bf16) or 1e-5 |ref| + 1e-7 (fp32), against the oracle on the
same logits; elements outside the rows must not change.
"""
from __future__ import annotations

import pytest
import torch

from oracle import linear_ce as oracle

pytestmark = pytest.mark.gpu


def _layout(rows, V, stride, offset, dtype, seed, dev):
    """(rows, V) logits at `stride` and `offset` elements in a buffer of NaN."""
    g = torch.Generator().manual_seed(seed)
    x = (torch.randn(rows, V, generator=g) * 4).to(dtype)
    buf = torch.full((offset + rows * stride + 64,), float("nan"), dtype=dtype, device=dev)
    view = buf[offset : offset + rows * stride].view(rows, stride)[:, :V]
    view.copy_(x)
    return x, buf, view


CASES = [
    # V, row stride, first element, dtype
    *[(V, V, off, torch.bfloat16) for V in (1, 7, 9, 2041, 2042, 2049) for off in (0, 1, 7)],
    (33, 40, 0, torch.bfloat16),       # aligned starts, ragged ends
    (2048, 2048, 3, torch.bfloat16),   # one chunk more than aligned
    (4097, 4097, 0, torch.bfloat16),
    (16383, 16385, 5, torch.bfloat16),
    (32769, 32769, 0, torch.bfloat16),
    (40955, 40955, 2, torch.bfloat16),
    (49153, 49160, 0, torch.bfloat16),
    (50257, 50304, 0, torch.bfloat16),
    (57344, 57344, 0, torch.bfloat16), # aligned, more than 16 chunks
    (65529, 65529, 0, torch.bfloat16), # the longest unaligned row in registers
    (65530, 65530, 0, torch.bfloat16), # one past it
    *[(V, V, off, torch.float32) for V in (3, 1021, 1025) for off in (0, 1, 3)],
    (32749, 32749, 0, torch.float32),
    (32766, 32767, 1, torch.float32),
]


@pytest.mark.parametrize("V,stride,offset,dtype", CASES)
def test_rows_of_any_alignment(V, stride, offset, dtype):
    from hlm_attn import ops

    dev = torch.device("cuda", 0)
    rows, n = 9, 11
    x, buf, view = _layout(rows, V, stride, offset, dtype, V + offset, dev)
    g = torch.Generator().manual_seed(1)
    targets = torch.randint(0, V, (rows,), generator=g)
    targets[0], targets[1], targets[2] = 0, V - 1, -100
    loss = ops.hip_linear_ce(view, targets.to(dev), n)
    torch.cuda.synchronize()
    rl, rg = oracle.ce_rows(x, targets, n)
    assert ((loss.double().cpu() - rl).abs() * n).max().item() <= 1e-4
    got, ref = view.double().cpu() * n, rg.double() * n
    rel, tol = (2.0**-8, 1e-6) if dtype == torch.bfloat16 else (1e-5, 1e-7)
    assert bool(((got - ref).abs() <= rel * ref.abs() + tol).all())
    inside = torch.zeros_like(buf, dtype=torch.bool)
    inside[offset : offset + rows * stride].view(rows, stride)[:, :V] = True
    assert bool(buf[~inside].isnan().all()), "an element outside the rows was written"


@pytest.mark.parametrize("V", [2048, 2049, 50257])
def test_infinite_and_nan_logits(V):
    """-inf logits get probability 0; +inf, NaN and an all -inf row make the
    row's loss NaN, and no other row's."""
    from hlm_attn import ops

    dev = torch.device("cuda", 0)
    x, _, view = _layout(6, V, V, 0, torch.bfloat16, 5, dev)
    for t in (x, view):
        t[1, ::2] = float("-inf")
        t[2, V - 1] = float("inf")
        t[3, 0] = float("nan")
        t[4] = float("-inf")
    targets = torch.full((6,), 1)
    loss = ops.hip_linear_ce(view, targets.to(dev), 6)
    torch.cuda.synchronize()
    rl, rg = oracle.ce_rows(x, targets, 6)
    assert loss.isnan().tolist() == [False, False, True, True, True, False]
    for r in (0, 1, 5):
        assert abs(loss[r].item() - rl[r].item()) * 6 <= 1e-4
        got, ref = view[r].double().cpu() * 6, rg[r].double() * 6
        assert bool(((got - ref).abs() <= 2.0**-8 * ref.abs() + 1e-6).all())
    assert bool((view[1, ::2] == 0).all())
