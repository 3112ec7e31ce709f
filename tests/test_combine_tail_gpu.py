"""The combine's gradient through autograd where some rows have no slot (capacity drops, the positional layout's
remainder): every row is written, the rows without a slot with zeros."""

from __future__ import annotations

import pytest
import torch

from gpu_util import dev

from moe_mi355 import ops
from moe_mi355.layer import CombineFn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,H,E,K,cap,layout", [
    (100, 72, 8, 3, 20, ops.LAYOUT_ROUTED),      # drops: rows past offsets[E]
    (33, 8, 7, 2, -1, ops.LAYOUT_REFERENCE),     # 66 rows in 7 chunks of 9: 3 left over
    (64, 264, 4, 1, -1, ops.LAYOUT_ROUTED),      # no row left over
    (50, 40, 16, 4, 0, ops.LAYOUT_ROUTED),       # every slot dropped: all rows
    (3, 16, 64, 1, -1, ops.LAYOUT_REFERENCE),    # fewer rows than experts: chunks of 0, all rows
])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
def test_rows_without_a_slot_are_zeros(N, H, E, K, cap, layout, dt):
    g = torch.Generator().manual_seed(N + H)
    idx = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(N)]).to(dev())
    p = ops.plan(idx, E, capacity=cap, layout=layout)
    y = torch.randn(N * K, H, generator=g).to(dt).to(dev()).requires_grad_(True)
    w = torch.rand(N, K, generator=g).to(dt).to(dev())
    dout = torch.randn(N, H, generator=g).to(dt).to(dev())
    torch.full((N * K, H), float("nan"), dtype=dt, device=dev())  # what the allocator hands out next
    (dy,) = torch.autograd.grad(CombineFn.apply(y, w, p), [y], dout)
    live = int(p.offsets[E])
    want = torch.zeros(N * K, H, dtype=torch.float64)
    rows = p.slot_row.cpu().long()
    keep = torch.ones(N * K, dtype=torch.bool) if p.drop is None else ~p.drop.cpu().reshape(-1)
    for s in range(N * K):
        if rows[s] < live and keep[s]:
            want[rows[s]] = w.cpu().double().reshape(-1)[s] * dout.cpu().double()[s // K]
    got = dy.cpu().double()
    assert bool((got[live:] == 0).all())
    # one product, rounded once to the type
    assert bool(((got - want).abs() <= (2.0**-8 if dt == torch.bfloat16 else 2.0**-24) * want.abs()).all())
