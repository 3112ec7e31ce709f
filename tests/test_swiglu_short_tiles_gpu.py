"""Tiles of at most 128 rows, in which half the waves of the row-grouped backward products idle (csrc/gemm.hip): a
row's result does not depend on how many rows its expert has beside it, so an expert of n rows has the bits of the first
n rows of the same expert with 256.  Sixteen experts and H = 4096 make 256 tiles of the products that may be split over
k, whole rounds that are not, so the order of every sum is the same too.  Both sides' numbers are tested against float64
where the products are."""

from __future__ import annotations

import pytest
import torch

from gpu_util import dev, say

from moe_mi355 import ops

pytestmark = pytest.mark.gpu

LENS = [1, 7, 31, 32, 33, 63, 64, 65, 96, 97, 120, 127, 128, 129, 200, 255]
H = 4096


def _inputs(F):
    g = torch.Generator(device=dev()).manual_seed(F)

    def randn(*s, std=1.0):
        return (torch.randn(*s, generator=g, device=dev()) * std).to(torch.bfloat16)

    E = len(LENS)
    full = torch.arange(E * 256, device=dev()).reshape(E, 256)
    rows = torch.cat([full[e, :n] for e, n in enumerate(LENS)])  # the short segments' rows among the full ones
    offs = torch.tensor([0] + LENS).cumsum(0).int().to(dev())
    offs_full = torch.arange(0, E * 256 + 1, 256, device=dev()).int()
    w = randn(E, F, H, std=H**-0.5), randn(E, F, H, std=H**-0.5), randn(E, H, F, std=F**-0.5)
    return randn(E * 256, H), randn(E * 256, H), w, rows, offs, offs_full


@pytest.mark.parametrize("F", [256, 160])
def test_bf16(F):
    say(f"[swiglu short tiles] bf16 F={F}")
    x, dy, w, rows, offs, offs_full = _inputs(F)
    keep = torch.zeros(x.shape[0], 1, dtype=torch.bool, device=dev())
    keep[rows] = True
    dy = torch.where(keep, dy, torch.zeros_like(dy))  # rows that only the full segments have add zeros to the weights'
    out = ops.swiglu_forward(x[rows], *w, offs)
    ref = ops.swiglu_forward(x, *w, offs_full)
    for a, b in zip(out, ref):
        assert torch.equal(a, b[rows])
    lean = ops.swiglu_forward(x[rows], *w, offs, keep_preact=False)
    assert torch.equal(lean[0], out[0]) and torch.equal(lean[2], out[2])
    got = ops.swiglu_backward(dy[rows], x[rows], out[0], out[1], *w, offs)
    want = ops.swiglu_backward(dy, x, ref[0], ref[1], *w, offs_full)
    assert torch.equal(got[0], want[0][rows])
    for a, b in zip(got[1:], want[1:]):
        assert torch.equal(a, b)


@pytest.mark.parametrize("F", [256, 192])
@pytest.mark.parametrize("keep_preact", [True, False])
def test_fp8(F, keep_preact):
    say(f"[swiglu short tiles] fp8 F={F} keep_preact={keep_preact}")
    x, _, w, rows, offs, offs_full = _inputs(F)
    q = [ops.quant_rows_fp8(t) for t in w]
    xq, sx = ops.quant_rows_fp8(x)
    wq, ws = tuple(t for t, _ in q), tuple(s for _, s in q)
    out = ops.swiglu_forward_fp8(xq[rows], sx[rows], wq, ws, offs, keep_preact=keep_preact)
    ref = ops.swiglu_forward_fp8(xq, sx, wq, ws, offs_full, keep_preact=keep_preact)
    for a, b in zip(out, ref):
        if a is not None:
            assert torch.equal(a, b[rows])
