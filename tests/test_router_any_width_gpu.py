"""The bf16 router kernels on hidden widths that are no multiple of their slices (64 and 256 columns), the few-token
forward, and the fp32 router with many experts: the parity checks of test_router_gpu.py at the edges of the slices,
chunks and token blocks."""

from __future__ import annotations

import pytest
import torch

from gpu_util import dev, say
import test_router_gpu as base

from moe_mi355 import _lib as L
from moe_mi355 import ops

pytestmark = pytest.mark.gpu

B, F = torch.bfloat16, torch.float32
SHAPES = [
    (37, 8, 8, 2, B, B),          # the narrowest: one 16-byte unit a row
    (70, 248, 8, 2, B, B),        # one partial 256-column slice
    (300, 264, 16, 4, B, B),      # a whole one and 8 columns of the next; waves without columns in the backward
    (1000, 1016, 32, 4, B, B),    # two expert tiles, the last wave's columns partial
    (9000, 712, 8, 3, B, B),      # 32 tokens a block in the forward
    (65, 2488, 64, 7, B, B),      # few-token forward, partial 64-column slice and 32-column chunk
    (5000, 1064, 64, 3, B, B),    # past the few-token forward: the wide form with a partial slice
    (4200, 72, 200, 4, B, B),     # 16 expert tiles, one whole slice and 8 columns
    (16, 40, 40, 2, B, B),        # H < 64 on the wide backward
    (130, 1144, 128, 12, B, B),
    (33, 2048, 256, 8, B, B),     # few tokens, 256 experts (K = 32 has candidates within the margin in 5% of tokens)
    (1, 64, 64, 8, B, B),
    (300, 1024, 128, 4, F, F),    # fp32, 8 expert tiles
    (9000, 132, 100, 4, F, F),    # fp32, several token groups a block, E % 16 != 0
    (257, 60, 256, 5, F, F),      # fp32, 16 expert tiles, H % 64 != 0
    (63, 516, 20, 3, F, F),       # fp32, two expert tiles in the backward
    (70, 68, 18, 2, F, F),        # fp32, E % 4 != 0: the generic backward
]


@pytest.mark.parametrize("shape", SHAPES, ids=base._ids)
def test_forward(shape):
    base.test_router_forward_parity(shape)


@pytest.mark.parametrize("shape", SHAPES, ids=base._ids)
@pytest.mark.parametrize("losses", [False, True], ids=["plain", "aux_z"])
def test_backward(shape, losses):
    base.test_router_backward_parity(shape, losses)


@pytest.mark.parametrize("N,H,E", [(100, 72, 8), (100, 520, 64), (40, 1096, 128)])
def test_neighbouring_rows_stay_out(N, H, E):
    """A partial slice must not read the next row: a NaN in one token changes nothing for the others, and the gate's
    last row nothing past it (the same call on the widened problem with zero columns gives the same logits)."""
    say(f"[router rows] N={N} H={H} E={E}")
    x, w, gw = base._inputs(N, H, E, 2, B, B, seed=H)
    ref = ops.router_forward(x.to(dev()), w.to(dev()), 2)[2]
    bad = x.clone()
    bad[N // 2] = float("nan")
    got = ops.router_forward(bad.to(dev()), w.to(dev()), 2)[2]
    rows = torch.arange(N) != N // 2
    assert torch.equal(got.cpu()[rows], ref.cpu()[rows])
    idx = torch.zeros(N, 2, dtype=torch.int64, device=dev())
    idx[:, 1] = 1
    dx0, _ = ops.router_backward(x.to(dev()), w.to(dev()), ref, idx, gw.to(dev()))
    dx1, _ = ops.router_backward(bad.to(dev()), w.to(dev()), ref, idx, gw.to(dev()))
    assert torch.equal(dx0, dx1)


def test_unaligned_gate_and_tokens():
    """Operands that are not 16-byte aligned take the general kernels and give the same routing."""
    N, H, E, K = 60, 96, 64, 4
    x, w, _ = base._inputs(N, H, E, K, B, B, seed=3)
    for off_x, off_w in ((0, 1), (1, 0)):
        xs = torch.empty(N * H + 8, dtype=B, device=dev())[off_x:off_x + N * H].view(N, H).copy_(x)
        ws = torch.empty(H * E + 8, dtype=B, device=dev())[off_w:off_w + H * E].view(H, E).copy_(w)
        assert (xs.data_ptr() | ws.data_ptr()) % 16
        base._check_forward(xs.cpu(), ws.cpu(), K)
        lib = L.load()
        assert lib.moe_router_fwd_workspace(N, H, E, K, 1, 1) > 0
        a = ops.router_forward(xs, ws, K)
        b = ops.router_forward(x.to(dev()), w.to(dev()), K)
        assert torch.equal(a[0], b[0])
        # 64 x 96 products: fp32 sums in another order
        assert float((a[2] - b[2]).abs().max()) <= 2 * H * 2.0**-24 * float((x.abs().float() @ w.abs().float()).max())


@pytest.mark.parametrize("H,E,K", [(264, 8, 2), (512, 8, 2), (1024, 8, 2), (264, 16, 4), (264, 5, 2), (96, 64, 4),
                                   (520, 128, 4)])
def test_unaligned_gate_backward(H, E, K):
    """A gate that starts off a 16-byte boundary: the router's and the norm-fused backward read it by element (E = 8, 16)
    or take the kernels that do.  The same bits where the same kernel runs; 32 < E: other kernels, whose dL/dlogits and
    results may each round the other way to bf16 (2^-8 of a value)."""
    N = 70
    x, w, gw = base._inputs(N, H, E, K, B, B, seed=11)
    ws = torch.empty(H * E + 8, dtype=B, device=dev())[1:1 + H * E].view(H, E).copy_(w)
    assert ws.data_ptr() % 16 == 2 and ws.is_contiguous()
    x, w, gw = x.to(dev()), w.to(dev()), gw.to(dev())
    idx, _, logits = ops.router_forward(x, w, K)[:3]
    a = ops.router_backward(x, w, logits, idx, gw)
    b = ops.router_backward(x, ws, logits, idx, gw)
    if E <= 32:
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    else:
        for p, q in zip(a, b):
            assert float((p.double() - q.double()).norm()) <= 2.0**-7 * float(p.double().norm())
    if E <= 16:
        nw, dxn = torch.ones(H, device=dev()), torch.randn(N, H, device=dev()).to(B)
        xn, rstd, idx, _, logits = ops.rmsnorm_router_forward(x, nw, 1e-5, w, K)[:5]
        a = ops.rmsnorm_router_backward(x, nw, rstd, xn, w, logits, idx, gw, dxn)
        b = ops.rmsnorm_router_backward(x, nw, rstd, xn, ws, logits, idx, gw, dxn)
        assert all(torch.equal(p, q) for p, q in zip(a, b))
