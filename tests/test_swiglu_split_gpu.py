"""Row-grouped products whose last round of tiles is split over k (csrc/gemm.hip, split_of): the split product against
the same call without room for its partial tiles, where the tiles run whole, and both against float64."""

from __future__ import annotations

import pytest
import torch

from gpu_util import TOL, assert_rel, dev, say

from moe_mi355 import _lib as L
from moe_mi355 import ops

pytestmark = pytest.mark.gpu



def _splits(counts, N, nk):
    """(whole tiles, tiles split, S) of each XCD of a row-grouped product N columns wide with nk k slices: the host's copy
    of the kernels' rule (split_parts, split_of and the tile ranges in csrc/gemm.hip)."""
    R, E, cols = sum(counts), len(counts), -(-N // 256)
    npart = min(64, 8 * -(-((-(-R // 256) + E) * cols) // 8))
    total = sum(-(-c // 256) for c in counts) * cols
    chunk, out = -(-total // 8), []
    for xcd in range(8):
        n = max(0, min(chunk, total - xcd * chunk))
        r, best, cost = n & 31, 1, nk
        for S in range(2, 9):
            if r * S > npart or S > nk:
                break
            c = ((r * S + 31) >> 5) * (-(-nk // S) + 20) + 5
            if c < cost:
                best, cost = S, c
        out.append((n - r, r, best if r else 1))
    return out


# (H, F, rows of each expert): one or several m-tiles an expert, ragged ones, k past and short of whole 64-wide slices,
# dxp's change of weights inside a slice (F % 64 == 32) and inside a part, a width that is no multiple of the tile,
# more tiles than a round (32 an XCD) and far fewer
CASES = [
    (256, 4096, [250, 250]),
    (264, 2080, [300, 1, 0, 256]),
    (512, 96, [700]),
    (1032, 3104, [257, 513, 40, 0]),
    (4096, 1056, [600] * 30),
    (1024, 2080, [20, 3, 0, 33]),  # few rows: dxp is split (the forward takes the few-row kernel)
    (4096, 4096, [4, 4]),
    # whole rounds and a few tiles more, which are split (33 to 36 tiles an XCD)
    (4096, 4096, [256 * 15, 300]),
    (4088, 4128, [256 * 14 + 100, 511]),
    (2048, 4160, [255] * 31 + [0, 500]),
]
ROUND_AND_PARTS = CASES[-3:]
# which of the down projection (y) and dxp (d) the rule splits in a case; the others run whole with the room for it as
# without, and with few rows the forward takes the few-row kernel instead
SPLIT = {(512, 96): "", (4096, 1056): "", (4096, 4096): "yd", (1024, 2080): "yd", (256, 4096): "yd", (264, 2080): "yd",
         (1032, 3104): "yd", (4088, 4128): "yd", (2048, 4160): "yd"}


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"H{c[0]}-F{c[1]}-E{len(c[2])}-R{sum(c[2])}")
def test_cases_split_what_they_say(case):
    H, Fd, counts = case
    y, d = _splits(counts, H, -(-Fd // 64)), _splits(counts, H, -(-2 * Fd // 64))
    for name, ranges in (("y", y), ("d", d)):
        assert any(S > 1 for _, _, S in ranges) == (name in SPLIT[(H, Fd)])
    if case in ROUND_AND_PARTS:
        assert any(S > 1 and full > 0 for full, _, S in y) and any(S > 1 and full > 0 for full, _, S in d)


def _call(fn, *args):
    L.check(fn(*args), "call")


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"H{c[0]}-F{c[1]}-E{len(c[2])}-R{sum(c[2])}")
def test_split_products(case):
    H, Fd, counts = case
    E, R = len(counts), sum(counts)
    say(f"[swiglu split] H={H} F={Fd} E={E} R={R}")
    lib = L.load()
    more = lib.moe_swiglu_split_workspace(R, H, Fd, E)
    assert more > 0
    g = torch.Generator(device=dev()).manual_seed(H + Fd + R)

    def randn(*s, std=1.0):
        return (torch.randn(*s, generator=g, device=dev()) * std).to(torch.bfloat16)

    xp, dy = randn(R, H), randn(R, H)
    wg, wu, wd = randn(E, Fd, H, std=H**-0.5), randn(E, Fd, H, std=H**-0.5), randn(E, H, Fd, std=Fd**-0.5)
    offs = torch.tensor([0] + counts).cumsum(0).int().to(dev())
    act, hgu, y = ops.swiglu_forward(xp, wg, wu, wd, offs)
    dxp, dwg, dwu, dwd = ops.swiglu_backward(dy, xp, act, hgu, wg, wu, wd, offs)
    # the same with the least workspace that the calls accept
    n = lib.moe_swiglu_workspace(E)
    ws = torch.empty(n, dtype=torch.uint8, device=dev())
    act0, hgu0, y0, dh, dxp0 = (torch.empty_like(t) for t in (act, hgu, y, hgu, dxp))
    s = L.stream_of(dev())
    p = [t.data_ptr() for t in (wg, wu, wd, offs)]
    _call(lib.moe_swiglu_fwd, xp.data_ptr(), *p, R, H, Fd, E, act0.data_ptr(), hgu0.data_ptr(), y0.data_ptr(),
          ws.data_ptr(), n, s)
    dws = [torch.empty_like(t) for t in (wg, wu, wd)]
    _call(lib.moe_swiglu_bwd, dy.data_ptr(), xp.data_ptr(), act0.data_ptr(), hgu0.data_ptr(), *p, R, H, Fd, E,
          dh.data_ptr(), dxp0.data_ptr(), *[t.data_ptr() for t in dws], ws.data_ptr(), n, s)
    torch.cuda.synchronize()
    assert torch.equal(act, act0) and torch.equal(hgu, hgu0)
    assert all(torch.equal(a, b) for a, b in zip((dwg, dwu, dwd), dws))
    # a product of n fp32 terms in any order is within n 2^-24 of the sum of their magnitudes, and rounds once to bf16
    for e in range(E):
        lo, hi = int(offs[e]), int(offs[e + 1])
        if lo == hi:
            continue
        a, d = act[lo:hi].double(), wd[e].double()
        h, w1 = dh[lo:hi].double(), torch.cat([wg[e], wu[e]]).double()
        for got, other, l, r in ((y, y0, a, d.t()), (dxp, dxp0, h, w1)):
            want = l @ r
            bound = 2.0**-8 * want.abs() + l.shape[1] * 2.0**-24 * (l.abs() @ r.abs()) + 1e-30
            for t in (got, other):
                assert bool(((t[lo:hi].double() - want).abs() <= bound).all())


def test_split_fp8():
    """The e4m3 down projection, split and whole: the same sums in another order, so within one bf16 rounding."""
    _fp8(1024, 4096, [300, 17, 0, 511])


def test_split_fp8_after_whole_rounds():
    H, Fd, counts = 4096, 8192, [256 * 15, 300]
    assert any(S > 1 and full > 0 for full, _, S in _splits(counts, H, Fd // 128))
    _fp8(H, Fd, counts)


@pytest.mark.parametrize("H,Fd,counts", [(4096, 8192, [4, 4]), (1040, 4128, [20, 3, 0, 33])])
def test_split_fp8_few_rows(H, Fd, counts):
    """The same with few rows, where the operation leaves it whole but a caller of the C ABI may pass the room."""
    _fp8(H, Fd, counts, room=True)


def _fp8(H, Fd, counts, room=False):
    E, R = len(counts), sum(counts)
    g = torch.Generator(device=dev()).manual_seed(7)
    ws = [torch.randn(E, Fd, H, generator=g, device=dev()) * H**-0.5, torch.randn(E, Fd, H, generator=g, device=dev())
          * H**-0.5, torch.randn(E, H, Fd, generator=g, device=dev()) * Fd**-0.5]
    q = [ops.quant_rows_fp8(t.to(torch.bfloat16)) for t in ws]
    xq, sx = ops.quant_rows_fp8(torch.randn(R, H, generator=g, device=dev()).to(torch.bfloat16))
    offs = torch.tensor([0] + counts).cumsum(0).int().to(dev())
    y = ops.swiglu_forward_fp8(xq, sx, tuple(t for t, _ in q), tuple(s for _, s in q), offs, keep_preact=False)[2]
    lib = L.load()
    assert lib.moe_swiglu_split_workspace(R, H, Fd, E) > 0
    n = lib.moe_swiglu_fwd_fp8_workspace(R, Fd, E)
    more = lib.moe_swiglu_split_workspace(R, H, Fd, E)
    wsp = torch.empty(n + more, dtype=torch.uint8, device=dev())
    y0 = torch.empty_like(y)
    for out, nbytes in ([(y, n + more)] if room else []) + [(y0, n)]:
        _call(lib.moe_swiglu_fwd_fp8, xq.data_ptr(), sx.data_ptr(), *[t.data_ptr() for pair in q for t in pair],
              offs.data_ptr(), R, H, Fd, E, None, None, out.data_ptr(), wsp.data_ptr(), nbytes, L.stream_of(dev()))
    torch.cuda.synchronize()
    a, b = y.double(), y0.double()
    # fp32 sums of 4096 terms differ by at most 2 x 4096 x 2^-24 of the sum of magnitudes, here below 8 rms of y
    assert bool(((a - b).abs() <= 2.0**-7 * b.abs() + 2 * Fd * 2.0**-24 * 8 * b.square().mean().sqrt() * Fd**0.5).all())


# fp32: a few tiles only, a last round after whole ones (64 blocks an XCD), column tiles that 8 XCDs share and not
F32_CASES = [
    (1000, 608, [300, 0, 140, 77]),
    (1024, 4096, [525, 503, 542, 471]),
    (260, 2080, [130, 1, 400]),
]


@pytest.mark.parametrize("case", F32_CASES, ids=lambda c: f"H{c[0]}-F{c[1]}-E{len(c[2])}")
def test_split_products_f32(case):
    H, Fd, counts = case
    E, R = len(counts), sum(counts)
    say(f"[swiglu split f32] H={H} F={Fd} E={E} R={R}")
    lib = L.load()
    assert lib.moe_swiglu_f32_split_workspace(R, H, Fd, E) > 0 and R > 64 * E
    g = torch.Generator(device=dev()).manual_seed(H + Fd + R)

    def randn(*s, std=1.0):
        return torch.randn(*s, generator=g, device=dev()) * std

    xp, dy = randn(R, H), randn(R, H)
    wg, wu, wd = randn(E, Fd, H, std=H**-0.5), randn(E, Fd, H, std=H**-0.5), randn(E, H, Fd, std=Fd**-0.5)
    offs = torch.tensor([0] + counts).cumsum(0).int().to(dev())
    act, hgu, y = ops.swiglu_forward(xp, wg, wu, wd, offs)
    dxp, dwg, dwu, dwd = ops.swiglu_backward(dy, xp, act, hgu, wg, wu, wd, offs)
    n = lib.moe_swiglu_f32_workspace(E)  # the least workspace: whole tiles
    ws = torch.empty(n, dtype=torch.uint8, device=dev())
    act0, hgu0, y0, dh, dxp0 = (torch.empty_like(t) for t in (act, hgu, y, hgu, dxp))
    s = L.stream_of(dev())
    p = [t.data_ptr() for t in (wg, wu, wd, offs)]
    _call(lib.moe_swiglu_fwd_f32, xp.data_ptr(), *p, R, H, Fd, E, act0.data_ptr(), hgu0.data_ptr(), y0.data_ptr(),
          ws.data_ptr(), n, s)
    dws = [torch.empty_like(t) for t in (wg, wu, wd)]
    _call(lib.moe_swiglu_bwd_f32, dy.data_ptr(), xp.data_ptr(), act0.data_ptr(), hgu0.data_ptr(), *p, R, H, Fd, E,
          dh.data_ptr(), dxp0.data_ptr(), *[t.data_ptr() for t in dws], ws.data_ptr(), n, s)
    torch.cuda.synchronize()
    # n fp32 terms in any order: within n 2^-24 of the sum of magnitudes; between two orders, twice that
    for e in range(E):
        lo, hi = int(offs[e]), int(offs[e + 1])
        if lo == hi:
            continue
        x, a, d = xp[lo:hi].double(), act[lo:hi].double(), wd[e].double()
        w1 = torch.cat([wg[e], wu[e]]).double()
        for got, other, l, r in ((hgu, hgu0, x, w1.t()), (y, y0, a, d.t()), (dxp, dxp0, dh[lo:hi].double(), w1)):
            want, mag = l @ r, l.abs() @ r.abs()
            bound = (l.shape[1] + 1) * 2.0**-24 * mag + 1e-30
            if got is y:  # each from its own act, which differs in rounding
                bound = bound + act0[lo:hi].double().sub(a).abs() @ r.abs()
            elif got is dxp:  # from dh of the whole tiles: the split's own differs by the rounding of dy . Wd
                bound = bound + (H + 16) * 2.0**-24 * 4 * mag
            for t in (got, other):
                assert bool(((t[lo:hi].double() - want).abs() <= bound).all())
        # the weights' gradients, from dh and act of the split products and of the whole ones
        gate, up = x @ wg[e].double().t(), x @ wu[e].double().t()
        sg = torch.sigmoid(gate)
        da = dy[lo:hi].double() @ d
        for got, whole, want in ((dwg[e], dws[0][e], (da * up * sg * (1 + gate * (1 - sg))).t() @ x),
                                 (dwu[e], dws[1][e], (da * gate * sg).t() @ x),
                                 (dwd[e], dws[2][e], dy[lo:hi].double().t() @ (gate * sg * up))):
            assert_rel(got, want, TOL[torch.float32], "dW")
            assert_rel(whole, want, TOL[torch.float32], "dW of whole tiles")
