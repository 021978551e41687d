"""The split count of a small forward grid (hlm_attn_fwd_split_count): shapes on
both sides of its rule, with and without a window (CPU), and the forward op at
the shapes that it splits more finely than one run per 12 key tiles (GPU),
against the fp32 oracle on the same bf16 inputs with the bounds of the split
forward's own tests: O |hip - ref| <= 1e-2 + 2e-2 |ref|, LSE 1e-3.
"""
from __future__ import annotations

import math

import pytest
import torch

from hlm_attn import _lib
from oracle import attention as oracle
from test_gpu_parity import make_inputs

POLICY = [
    # B, T, H, D, window, splits
    (1, 960, 4, 64, 0, 1),       # 15 key tiles
    (1, 1024, 4, 64, 0, 3),      # 16: three runs of at least five
    (1, 1024, 8, 64, 0, 1),      # as many workgroups as four times the key tiles
    (1, 1500, 4, 64, 0, 4),
    (1, 1025, 6, 128, 0, 3),
    (1, 2000, 4, 128, 1024, 3),  # windowed, few units
    (1, 2047, 12, 64, 1024, 1),  # windowed, the chip is busy enough
    (1, 6000, 8, 64, 3000, 1),
    (1, 4000, 12, 64, 0, 2),     # half of the slots taken, long rows
    (1, 4000, 16, 64, 0, 1),
    (1, 4000, 12, 128, 0, 2),
    (2, 1777, 12, 128, 0, 1),
    (1, 65536, 1, 128, 0, 1),    # as many workgroups as slots
    (1, 1 << 30, 1, 64, 0, 1),
]


@pytest.mark.parametrize("B,T,H,D,window,splits", POLICY)
def test_split_count(B, T, H, D, window, splits):
    assert _lib.load().hlm_attn_fwd_split_count(B, T, H, D, window) == splits


@pytest.mark.gpu
@pytest.mark.parametrize("B,T,H,Hkv,D,window", [(1, 1024, 4, 4, 64, 0), (1, 1500, 4, 1, 64, 0), (1, 1025, 6, 2, 128, 0),
                                                (1, 2000, 4, 4, 128, 1024), (2, 1037, 2, 2, 64, 1001)])
def test_forward_op_in_short_runs_matches_the_oracle(B, T, H, Hkv, D, window):
    from hlm_attn import ops

    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    assert _lib.load().hlm_attn_fwd_split_count(B, T, H, D, window) >= 3
    print(f"case short runs B={B} T={T} H={H} Hkv={Hkv} D={D} W={window}", flush=True)
    q, k, v, _ = make_inputs(B, T, H, Hkv, D, 90 + T)
    o, lse = ops.hip_attn_fwd(q.cuda(), k.cuda(), v.cuda(), window, 1.0 / math.sqrt(D))
    ro, rlse = oracle.forward(q, k, v, window or None)
    assert bool(((o.float().cpu() - ro).abs() <= 1e-2 + 2e-2 * ro.abs()).all())
    assert (lse.cpu() - rlse).abs().max().item() <= 1e-3
