"""The backward with long dQ and dK/dV tiles cut into chunks
(hlm_attn_bwd_split): its argument checks and the shapes it applies to (CPU),
and its results against hlm_attn_bwd and the fp32 oracle (GPU).

The gradients are the same fp32 products summed in another order and rounded
to bf16 once, so two results differ by at most one bf16 step of the value
(2^-7 relative) plus the fp32 sums' own reordering error, which is far below
1e-5 of the largest gradient.  Where only one of dQ and dK/dV is cut, the
other one's kernel is the same and its result bit-identical.  Every call
starts from a NaN-filled workspace.
"""
from __future__ import annotations

import ctypes
import math

import pytest
import torch

from hlm_attn import _lib
from oracle import attention as oracle
from test_gpu_parity import assert_grad, make_inputs

CASES = [
    # B, T, H, Hkv, D, window: dK/dV cut, dQ as the sizes have it
    (1, 1, 64, 1, 64, None),      # one token, one key tile, 64 query heads: chunks of whole heads
    (1, 1000, 8, 2, 64, 200),     # 44 query tiles a key tile
    (1, 129, 32, 1, 128, None),   # a second key tile of one row
    (1, 333, 4, 1, 64, 129),      # few tokens, four heads to a key tile
    (1, 128, 16, 2, 64, None),    # one key tile
    (1, 300, 40, 2, 64, 40),      # short window, many heads: chunks end inside a head
    (1, 777, 16, 1, 128, None),   # ragged, causal: key tiles with 1 to 16 chunks
    (2, 1025, 12, 4, 64, None),
    (1, 1500, 8, 2, 128, 700),    # windowed: the rotated tile order across chunks
    (2, 1777, 12, 4, 128, None),
    (1, 2048, 6, 6, 64, None),    # no grouping
]
DQ_CASES = [
    # dQ cut
    (1, 1000, 4, 4, 128, None),   # ragged, two chunks
    (1, 2048, 1, 1, 64, None),    # chunks of the shortest length
    (2, 2049, 2, 2, 64, None),    # a last query tile of one row
    (1, 2945, 2, 1, 64, 1944),    # windowed, and the ragged last query tile lacks the last chunk
    (1, 3201, 2, 2, 128, 2000),
    (1, 8192, 1, 1, 64, None),    # 16 chunks, the largest number
]


def _bytes(B, T, H, Hkv, D, window):
    return _lib.load().hlm_attn_bwd_split_workspace_bytes(B, T, H, Hkv, D, window or 0)


@pytest.mark.parametrize("case", CASES + DQ_CASES)
def test_split_applies_to_the_cases_below(case):
    B, T, H, Hkv, D, _ = case
    tiles, n = (T + 127) // 128, _bytes(*case)
    # One chunk of every (batch, kv head), fp32 dK and dV of 128 keys, or of every (batch, head), fp32 dQ.
    kv_block, q_block = B * Hkv * 128 * D * 8, B * H * 128 * D * 4
    assert any(n % b == 0 and 2 * b <= n <= 16 * tiles * b for b in (kv_block, q_block))
    assert n // (128 * D * 8) <= 256 * (3 if D == 64 else 2), "at most one filling of the chip"


@pytest.mark.parametrize(
    "case",
    [
        (8, 2048, 12, 12, 64, 512),    # the chip is full
        (1, 16384, 16, 16, 128, 2048),
        (1, 1000, 6, 6, 64, 300),      # short rows
        (1, 480, 6, 6, 64, None),
        (2, 1000, 8, 4, 64, 256),
        (1, 4096, 16, 16, 64, None),   # chunks would be as long as the slots they fill are slow
        (1, 4096, 8, 8, 128, 1024),
        (0, 128, 2, 2, 64, None),
    ],
)
def test_split_does_not_apply(case):
    assert _bytes(*case) == 0


def test_split_backward_checks_its_workspace():
    lib = _lib.load()
    assert lib.hlm_attn_bwd_split_workspace_bytes(1, 128, 3, 2, 64, 0) == -1
    assert lib.hlm_attn_bwd_split_workspace_bytes(1, 128, 2, 2, 96, 0) == -2
    T, H, D = 129, 32, 128
    need = _bytes(1, T, H, 1, D, None)
    s, p = (ctypes.c_int64 * 3)(T * H * D, H * D, D), ctypes.c_void_p(0x1000)

    def call(ws, n):
        return lib.hlm_attn_bwd_split(*([p] * 10), ws, n, 1, T, H, 1, D, *([s] * 8), 0, 0.1, None)

    assert call(None, need) == -1 and b"partial workspace" in lib.hlm_attn_last_error()
    assert call(ctypes.c_void_p(0x1008), need) == -1
    assert call(p, need - 1) == -1 and b"needed" in lib.hlm_attn_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES + DQ_CASES)
def test_split_backward_matches_the_unsplit_one_and_the_oracle(case):
    from hlm_attn import ops

    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    dev = torch.device("cuda", 0)
    B, T, H, Hkv, D, window = case
    print(f"case split B={B} T={T} H={H} Hkv={Hkv} D={D} W={window}", flush=True)
    q, k, v, do = make_inputs(B, T, H, Hkv, D, 70 + T)
    qd, kd, dod = (t.to(dev) for t in (q, k, do))
    vd = torch.empty(B, T, 2 * Hkv, D, dtype=torch.bfloat16, device=dev)[:, :, Hkv:]  # a strided view
    vd.copy_(v)
    w, scale, lib = window or 0, 1.0 / math.sqrt(D), _lib.load()
    o, lse = ops.hip_attn_fwd(qd, kd, vd, w, scale)
    n = _bytes(*case)
    got = []
    for split in (False, True, True):
        dq, dk, dv = (torch.full_like(t, float("nan"), memory_format=torch.contiguous_format) for t in (qd, kd, vd))
        delta = torch.empty(2 * B * H * T, device=dev)
        part = torch.full((n // 4,), float("nan"), device=dev)
        ptrs = [t.data_ptr() for t in (qd, kd, vd, o, dod, lse, dq, dk, dv, delta)]
        st = [_lib.strides3(t) for t in (qd, kd, vd, o, dod, dq, dk, dv)]
        tail = (B, T, H, Hkv, D, *st, w, scale, ops._stream_handle(dev))
        if split:
            rc = lib.hlm_attn_bwd_split(*ptrs, part.data_ptr(), n, *tail)
        else:
            rc = lib.hlm_attn_bwd(*ptrs, *tail)
        _lib.check(rc, lib)
        torch.cuda.synchronize()
        got.append((dq, dk, dv))
    one, two, again = got
    # By the sizes, the first cases cut dK/dV only and the others dQ or both.
    assert torch.equal(one[0], two[0]) == (case in CASES[:9])
    assert all(torch.equal(a, b) for a, b in zip(two, again)), "not deterministic"
    for name, a, b in zip(("dq", "dk", "dv"), one, two):
        a, b = a.float(), b.float()
        assert bool(((a - b).abs() <= 2.0**-7 * a.abs() + 1e-5 * a.abs().max()).all()), name
    via_op = ops.hip_attn_bwd(dod, qd, kd, vd, o, lse, w, scale)
    assert all(torch.equal(a, b) for a, b in zip(two, via_op)), "the op takes the split path"
    if H * T <= 16 * 1024:
        rdq, rdk, rdv = oracle.backward(q, k, v, do, window)
        for name, a, r in zip(("dq", "dk", "dv"), two, (rdq, rdk, rdv)):
            assert_grad(name, a.float().cpu(), r)


def _inputs(case, dev):
    from hlm_attn import ops

    B, T, H, Hkv, D, window = case
    q, k, v, do = (t.to(dev) for t in make_inputs(B, T, H, Hkv, D, 70 + T))
    w, scale = window or 0, 1.0 / math.sqrt(D)
    o, lse = ops.hip_attn_fwd(q, k, v, w, scale)
    return q, k, v, do, o, lse, w, scale


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[1], CASES[6], CASES[9], DQ_CASES[0], DQ_CASES[3], DQ_CASES[4]])
def test_split_backward_reads_and_writes_any_strides(case):
    """q, k, v as views of one projection, dO and o as (B, H, T, D), dq, dk and dv
    into views of one gradient: bit-identical to contiguous tensors, and
    nothing else in the buffers is written."""
    from hlm_attn import ops

    dev = torch.device("cuda", 0)
    B, T, H, Hkv, D, _ = case
    print(f"case split strides {case}", flush=True)
    q, k, v, do, o, lse, w, scale = _inputs(case, dev)
    want = ops.hip_attn_bwd(do, q, k, v, o, lse, w, scale)

    def views(fill):
        buf = torch.full((B, T, H + 2 * Hkv + 1, D), fill, dtype=torch.bfloat16, device=dev)
        return buf, (buf[:, :, :H], buf[:, :, H : H + Hkv], buf[:, :, H + Hkv : -1])

    _, ins = views(float("nan"))
    for dst, src in zip(ins, (q, k, v)):
        dst.copy_(src)
    do_t, o_t = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (do, o))
    gbuf, grads = views(7.0)
    delta = torch.empty(2 * B * H * T, device=dev)
    n = _bytes(*case)
    part = torch.full((n // 4,), float("nan"), device=dev)
    lib = _lib.load()
    rc = lib.hlm_attn_bwd_split(*(t.data_ptr() for t in (*ins, o_t, do_t, lse, *grads, delta, part)), n, B, T, H, Hkv, D,
                                *(_lib.strides3(t) for t in (*ins, o_t, do_t, *grads)), w, scale, ops._stream_handle(dev))
    _lib.check(rc, lib)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(grads, want))
    assert bool((gbuf[:, :, -1] == 7).all())


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[1], DQ_CASES[0], (1, 1500, 4, 2, 64, None)])
def test_split_backward_in_a_graph(case):
    """Forward and backward captured in a HIP graph, the workspace in its pool,
    and replayed with eager work between: every replay equals the eager result."""
    from hlm_attn import ops

    dev = torch.device("cuda", 0)
    print(f"case split graph {case}", flush=True)
    q, k, v, do, _, _, w, scale = _inputs(case, dev)

    def step():
        o, lse = ops.hip_attn_fwd(q, k, v, w, scale)
        return (o, lse, *ops.hip_attn_bwd(do, q, k, v, o, lse, w, scale))

    eager = [t.clone() for t in step()]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        static = step()
    for replay in range(3):
        for t in static:
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(static, eager)), f"replay {replay}"
        step()  # the eager pool's workspace, of the same size
        torch.cuda.synchronize()
