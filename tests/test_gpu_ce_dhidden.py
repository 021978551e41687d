"""hlm_ce_dhidden, the LM head's dhidden product with the vocabulary split over
workgroups: its checks and rule (CPU) and its results (GPU).

The product is compared with the float64 product of the same bf16 operands:
one bf16 rounding of the result (2^-8 relative) plus the fp32 sums' error,
which is at most K * 2^-24 of the sum of absolute products.  Around the
operands lie NaNs, which no result may see.
"""
from __future__ import annotations

import ctypes

import pytest
import torch

from hlm_attn import _lib

CASES = [
    # rows, hidden, vocab
    (1, 8, 1),
    (3, 16, 63),
    (255, 64, 64),
    (256, 256, 65),
    (257, 264, 512),       # a second row tile of one row, a second column tile of 8
    (300, 248, 1000),
    (40, 768, 1025),       # 17 steps: runs of unequal length
    (512, 320, 4099),
    (904, 768, 5000),
    (2048, 1024, 2000),
    (130, 512, 50257),
    (8192, 768, 600),      # more tiles than half the chip: runs of one or two
]


def test_rule_and_workspace():
    lib = _lib.load()
    pays, nbytes = lib.hlm_ce_dhidden_pays, lib.hlm_ce_dhidden_workspace_bytes
    assert pays(4096, 768, 32768) == 1 and nbytes(4096, 768, 32768) == 5 * 48 * 256 * 256 * 4
    assert pays(904, 768, 50257) == 1
    # K has to be long, longer where there are more tiles, however few CUs the library's product takes
    assert pays(272, 256, 3968) == 0 and pays(272, 256, 3969) == 1 and pays(300, 256, 1000) == 0
    assert pays(8192, 256, 3969) == 1 and pays(8193, 256, 3969) == 0  # 32 tiles, 33
    assert pays(4096, 2048, 5952) == 0 and pays(4096, 2048, 5953) == 1  # 128 tiles
    assert pays(5600, 1024, 900) == 0 and pays(8192, 768, 600) == 0 and pays(8192, 768, 1000) == 0
    assert pays(8192, 768, 32768) == 0  # 96 tiles: two runs fill 192 CUs
    assert pays(16384, 768, 32768) == 0  # the chip is full without a split
    assert pays(4096, 772, 32768) == 0 and pays(0, 768, 32768) == 0  # not taken
    assert nbytes(1, 8, 1) == 0 and nbytes(0, 768, 32768) == 0
    assert nbytes(4096, 772, 32768) == -2 and nbytes(-1, 768, 100) == -1
    for rows, hidden, vocab in CASES:
        tiles = -(-rows // 256) * -(-hidden // 256)
        runs = nbytes(rows, hidden, vocab) // (tiles * 256 * 256 * 4)
        assert runs == 0 or (2 <= runs <= 256 // tiles and 8 * runs <= -(-vocab // 64))


def test_arguments_are_checked_before_touching_the_device():
    lib = _lib.load()
    p = ctypes.c_void_p(0x1000)

    def call(g=p, ldg=1024, w=p, ldw=768, c=p, ldc=768, M=300, N=768, K=1000, ws=p, n=1 << 30):
        return lib.hlm_ce_dhidden(g, ldg, w, ldw, c, ldc, M, N, K, ws, n, None)

    for bad in (dict(ldg=1000), dict(ldg=1025), dict(ldw=760), dict(ldw=769), dict(ldc=760), dict(ldc=772), dict(g=None),
                dict(w=ctypes.c_void_p(0x1008)), dict(c=None), dict(ws=None), dict(n=16), dict(M=-1), dict(K=0)):
        assert call(**bad) == -1, bad
    assert call(N=772, ldw=776, ldc=776) == -2
    assert call(M=0) == 0


@pytest.mark.parametrize("vocab", [2097088, 2097089, 2097152, 2097153])
def test_the_rule_and_the_stride_check_agree_at_the_longest_vocabularies(vocab):
    """Where the rule says yes, the loss's workspace rows (a multiple of 64, and
    64 more where that is a multiple of 4 KB) are taken."""
    lib = _lib.load()
    stride = -(-vocab // 64) * 64
    stride += 64 * (stride * 2 % 4096 == 0)
    p = ctypes.c_void_p(0x1000)
    rc = lib.hlm_ce_dhidden(p, stride, p, 64, p, 64, 0, 64, vocab, p, 1 << 40, None)
    assert (rc == 0) == (lib.hlm_ce_dhidden_pays(1, 64, vocab) == 1) == (vocab <= 1 << 21), lib.hlm_attn_last_error()


def test_op_leaves_strides_that_the_kernel_refuses_to_the_library(monkeypatch):
    """The row stride of a single row may be anything, also below its length."""
    from hlm_attn import ops

    class OnDevice(torch.Tensor):
        is_cuda = True

    def row(cols, stride):
        return torch.zeros(64, dtype=torch.bfloat16).as_strided((1, cols), (stride, 1)).as_subclass(OnDevice)

    monkeypatch.setattr(_lib.load(), "hlm_ce_dhidden_pays", lambda *a: 1)
    assert ops._ce_dhidden_ready(row(64, 64), row(32, 32), 1, row(32, 32))
    for strides in ((8, 32, 32), (64, 0, 32), (64, 8, 32), (64, 32, 24), (64, 1 << 23, 32), (1 << 22, 32, 32)):
        work, weight, out = (row(c, s) for c, s in zip((64, 32, 32), strides))
        assert not ops._ce_dhidden_ready(work, weight, 1, out), strides


@pytest.mark.gpu
@pytest.mark.parametrize("rows,hidden,vocab", CASES)
def test_matches_the_product_of_the_same_operands(rows, hidden, vocab):
    from hlm_attn import ops

    dev = torch.device("cuda", 0)
    print(f"case rows={rows} hidden={hidden} vocab={vocab}", flush=True)
    lib = _lib.load()
    gen = torch.Generator(device=dev).manual_seed(rows + vocab)
    padded = -(-vocab // 64) * 64
    g_all = torch.full((rows + 2, padded + 8), float("nan"), dtype=torch.bfloat16, device=dev)
    g = g_all[:rows, :padded]
    g[:, :vocab] = (torch.rand(rows, vocab, generator=gen, device=dev) - 0.5).bfloat16()
    g[:, vocab:] = 0
    w_all = torch.full((vocab + 2, hidden + 16), float("nan"), dtype=torch.bfloat16, device=dev)
    w = w_all[:vocab, :hidden]
    w.copy_((torch.randn(vocab, hidden, generator=gen, device=dev) * 0.05).bfloat16())
    ref = g[:, :vocab].double() @ w.double()
    mag = g[:, :vocab].double().abs() @ w.double().abs()
    out = []
    for _ in range(2):
        c_all = torch.full((rows + 1, hidden + 8), 7.0, dtype=torch.bfloat16, device=dev)
        n = lib.hlm_ce_dhidden_workspace_bytes(rows, hidden, vocab)
        ws = torch.full((max(n // 4, 4),), float("nan"), device=dev)
        rc = lib.hlm_ce_dhidden(g.data_ptr(), g.stride(0), w.data_ptr(), w.stride(0), c_all.data_ptr(), c_all.stride(0),
                                rows, hidden, vocab, ws.data_ptr(), n, ops._stream_handle(dev))
        _lib.check(rc, lib)
        torch.cuda.synchronize()
        assert bool((c_all[rows:] == 7).all()) and bool((c_all[:, hidden:] == 7).all())
        out.append(c_all[:rows, :hidden].clone())
    assert torch.equal(*out), "not deterministic"
    err = (out[0].double() - ref).abs()
    assert bool((err <= 2.0**-8 * ref.abs() + vocab * 2.0**-24 * mag).all())


@pytest.mark.gpu
@pytest.mark.parametrize("rows,hidden,vocab,stride", [(300, 256, 1000, 1024), (300, 256, 4000, 4032), (300, 260, 1000, 1024), (4096, 2304, 128, 128)])
def test_op_takes_either_product(rows, hidden, vocab, stride):
    """The op gives the same result where the kernel applies and where the
    library's product runs (hidden no multiple of 8; too many tiles)."""
    from hlm_attn import ops

    dev = torch.device("cuda", 0)
    gen = torch.Generator(device=dev).manual_seed(3)
    work = torch.zeros(rows, stride, dtype=torch.bfloat16, device=dev)
    work[:, :vocab] = torch.rand(rows, vocab, generator=gen, device=dev).bfloat16()
    weight = torch.randn(vocab, hidden, generator=gen, device=dev).bfloat16()
    out = torch.empty(rows, hidden, dtype=torch.bfloat16, device=dev)
    ops.hip_ce_dhidden(work, weight, vocab, out)
    ref = work[:, :vocab].double() @ weight.double()
    assert ((out.double() - ref).norm() / ref.norm()).item() <= 2.0**-8
    with pytest.raises(RuntimeError, match="do not match"):
        ops.hip_ce_dhidden(work, weight, vocab - 1, out)
