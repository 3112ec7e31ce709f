"""The forward products for few rows per expert (csrc/gemm_small.hip): segments at the edges of the 16-, 32- and 64-row
passes, rows of one partial 128-byte chunk and of many, both column widths of a block, against float64."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from gpu_util import dev, say

from moe_mi355 import ops

pytestmark = pytest.mark.gpu

# (dtype, H, F, rows of each expert): the average stays within the path's rule (24 rows bf16, 32 fp32)
CASES = [
    ("bf16", 8, 32, [1]),  # one partial chunk, the least of every size
    ("bf16", 136, 96, [5, 0, 17, 64, 3, 70, 0, 8, 1, 2]),  # empty experts, several passes, H % 64 != 0
    ("bf16", 1000, 608, [16, 15, 0, 33, 32, 31]),
    ("bf16", 520, 8256, [1, 3]),  # more than 512 blocks of the gate/up product only
    ("bf16", 4104, 64, [2, 0, 1, 1, 0, 0, 0, 3] * 16),
    ("f32", 4, 32, [3]),
    ("bf16", 64, 64, [0] * 70 + [300] + [0, 33] * 40),  # most rows on one expert past the first 64
    ("f32", 1004, 160, [0, 65, 100, 1, 16, 9]),
    ("f32", 132, 4128, [1, 17, 32, 48]),
    ("bf16", 200, 96, [34, 48, 49, 63, 65, 128, 129, 1] + [0] * 20),  # 64-row passes: partial, whole, several
    ("bf16", 1032, 4128, [50, 0, 0, 0, 66, 0, 0]),  # ... over many columns: 64 weight rows a block
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-H{c[1]}-F{c[2]}-{sum(c[3])}rows")
def test_few_rows(case):
    name, H, Fd, counts = case
    say(f"[swiglu small] {case[:3]} counts={counts[:10]}")
    dt = torch.bfloat16 if name == "bf16" else torch.float32
    E, R = len(counts), sum(counts)
    assert R <= (24 if name == "bf16" else 32) * E
    g = torch.Generator().manual_seed(H + Fd + R)
    tail = 3  # rows past offsets[E]: not computed
    xp = torch.randn(R + tail, H, generator=g).to(dt)
    wg, wu = ((torch.randn(E, Fd, H, generator=g) / H**0.5).to(dt) for _ in range(2))
    wd = (torch.randn(E, H, Fd, generator=g) / Fd**0.5).to(dt)
    offs = torch.tensor([0] + counts, dtype=torch.int32).cumsum(0).int()
    args = [t.to(dev()) for t in (xp, wg, wu, wd, offs)]
    act, hgu, y = ops.swiglu_forward(*args)
    act2, none, y2 = ops.swiglu_forward(*args, keep_preact=False)
    assert none is None and torch.equal(act[:R], act2[:R]) and torch.equal(y[:R], y2[:R])
    # bounds: u = the type's unit roundoff; fp32 sums of n terms err by at most n u32 of the sum of magnitudes, and a
    # result rounds once; silu has a slope of at most 1.1, so errors dg, du of the pre-activations give act at most
    # 1.1 |u| dg + |silu(g)| du plus its own rounding and the hardware sigmoid's few ulp of fp32
    u32 = 2.0**-24
    u = 2.0**-8 if name == "bf16" else u32  # significands of 8 and 24 bits
    for e in range(E):
        lo, hi = int(offs[e]), int(offs[e + 1])
        if lo == hi:
            continue
        x, a, b, d = (t.double() for t in (xp[lo:hi], wg[e], wu[e], wd[e]))
        gg, uu = x @ a.t(), x @ b.t()
        dg = u * gg.abs() + (H + 4) * u32 * (x.abs() @ a.abs().t()) + 1e-30
        du = u * uu.abs() + (H + 4) * u32 * (x.abs() @ b.abs().t()) + 1e-30
        hg = hgu[lo:hi].cpu().double()
        assert bool(((hg[:, :Fd] - gg).abs() <= dg).all()) and bool(((hg[:, Fd:] - uu).abs() <= du).all())
        s = F.silu(gg)
        da = 1.1 * (uu.abs() + du) * dg + s.abs() * du + (u + 16 * u32) * (s * uu).abs() * (1 + 4 * u) + 1e-30
        got = act[lo:hi].cpu().double()
        assert bool(((got - s * uu).abs() <= da).all())
        yy = got @ d.t()  # the down projection of the act it was given
        dy = u * yy.abs() + (Fd + 4) * u32 * (got.abs() @ d.abs().t()) + 1e-30
        assert bool(((y[lo:hi].cpu().double() - yy).abs() <= dy).all())


@pytest.mark.parametrize("name,H,Fd", [("bf16", 1032, 2080), ("f32", 516, 1056)])
def test_rows_do_not_depend_on_their_neighbours(name, H, Fd):
    """An expert's rows have the same bits whatever the other experts' rows are, and wherever in the expert's own rows
    they lie: the first, a later and a partial 32-row pass, with passes of other experts ahead of them or none."""
    say(f"[swiglu small] neighbours {name} H={H} F={Fd}")
    dt = torch.bfloat16 if name == "bf16" else torch.float32
    E = 12
    g = torch.Generator().manual_seed(H)
    wg, wu = ((torch.randn(E, Fd, H, generator=g) / H**0.5).to(dt).to(dev()) for _ in range(2))
    wd = (torch.randn(E, H, Fd, generator=g) / Fd**0.5).to(dt).to(dev())
    rows = torch.randn(70, H, generator=g).to(dt).to(dev())  # expert 7's

    def run(before, own, after):
        counts = [0] * E
        counts[2], counts[7], counts[9] = before, own.shape[0], after
        assert sum(counts) <= 16 * E
        other = torch.randn(before + after, H, device=dev()).to(dt)
        xp = torch.cat([other[:before], own, other[before:]])
        offs = torch.tensor([0] + counts).cumsum(0).int().to(dev())
        return [t[before:before + own.shape[0]] for t in ops.swiglu_forward(xp, wg, wu, wd, offs)]

    want = run(0, rows, 0)
    for before, after in ((65, 0), (100, 20), (1, 33)):
        assert all(torch.equal(a, b) for a, b in zip(run(before, rows, after), want))
    part = run(40, rows[37:], 3)  # the same rows as others of the segment
    assert all(torch.equal(a, b[37:]) for a, b in zip(part, want))
