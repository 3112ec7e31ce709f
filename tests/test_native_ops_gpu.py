"""The operations bound in csrc/torch_router.cpp take every form that their Python callers may pass: strided views and
narrower index types give the bits of the contiguous call, what has the wrong rank, type or device is refused, and no
tokens at all give empty results.  Every kernel's numbers are tested where its sizes are."""

import pytest
import torch

from moe_mi355 import ops

pytestmark = pytest.mark.gpu
N, H, E, K, F = 37, 72, 8, 2, 64


def strided(t):
    """The same values in a tensor whose rows are not packed."""
    wide = torch.empty(*t.shape[:-1], t.shape[-1] * 2, dtype=t.dtype, device=t.device)
    view = wide[..., ::2]
    view.copy_(t)
    assert not view.is_contiguous()
    return view


def same(a, b):
    for s, t in zip(a, b):
        assert (s is None and t is None) or torch.equal(s, t)


@pytest.fixture
def data():
    g = torch.Generator(device="cuda").manual_seed(5)

    def rnd(*shape, dtype=torch.bfloat16):
        return torch.randn(*shape, generator=g, device="cuda").to(dtype)

    return rnd


def routed(rnd, dtype):
    x, gw, nw = rnd(N, H, dtype=dtype), rnd(H, E, dtype=dtype), rnd(H, dtype=dtype)
    return x, gw, nw, ops.rmsnorm_router_forward(x, nw, 1e-6, gw, K, None, 0.01, 0.001)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_strided_inputs_give_the_contiguous_bits(data, dtype):
    x, gw, nw, fwd = routed(data, dtype)
    bias = data(E, dtype=torch.float32)
    same(ops.router_forward(strided(x), strided(gw), K, strided(bias)), ops.router_forward(x, gw, K, bias))
    assert ops.router_forward(x, gw, K, w_dtype=torch.float32)[1].dtype == torch.float32
    same(ops.rmsnorm_router_forward(strided(x), strided(nw), 1e-6, strided(gw), K, None, 0.01, 0.001), fwd)
    xn, rstd, idx, w, logits, _, cnt = fwd[:7]
    gwt, dxn = data(N, K, dtype=dtype), data(N, H, dtype=dtype)
    g1 = torch.ones((), device=x.device)

    def bwd(f):
        return ops.rmsnorm_router_backward(f(x), f(nw), rstd, f(xn), f(gw), f(logits), f(idx), f(gwt), f(dxn), cnt, g1, g1,
                                           0.01, 0.001)

    same(bwd(strided), bwd(lambda t: t))
    for capacity in (-1, 5):
        p = ops.plan(idx, E, capacity)
        q = ops.plan(strided(idx).int(), E, capacity)
        if capacity < 0:
            assert p.drop is None and q.drop is None
        kept = int(p.offsets[-1])
        same((p.drop, p.offsets, p.ndrop, p.slot_row), (q.drop, q.offsets, q.ndrop, q.slot_row))
        xp = ops.permute(x, p)
        assert torch.equal(xp[:kept], ops.permute(strided(x), p)[:kept])
        y = data(p.rows, H, dtype=dtype)
        assert torch.equal(ops.combine(y, w, p), ops.combine(strided(y), strided(w), p))
        for need_dw in (True, False):
            same(ops.combine_backward(dxn, y, w, p, need_dw, zero_tail=True),
                 ops.combine_backward(strided(dxn), y, strided(w), p, need_dw, zero_tail=True))
        assert torch.equal(ops.unpermute_sum(y, p, dxn), ops.unpermute_sum(strided(y), p, strided(dxn)))


def test_what_was_refused_stays_refused(data):
    x, gw, nw, fwd = routed(data, torch.bfloat16)
    xn, rstd, idx, w, logits, _, cnt = fwd[:7]
    p = ops.plan(idx, E)
    wg, wd = data(E, F, H), data(E, H, F)
    xp = ops.permute(x, p)
    act, hgu, y = ops.swiglu_forward(xp, wg, wg, wd, p.offsets)
    assert ops.swiglu_forward(xp, wg, wg, wd, p.offsets, keep_preact=False)[1] is None
    for bad in (lambda: ops.router_forward(x[None], gw, K), lambda: ops.router_forward(x[:, :64], gw, K),
                lambda: ops.rmsnorm_router_backward(x[None], nw, rstd, xn, gw, logits, idx, w, None, cnt),
                lambda: ops.plan(idx.reshape(-1), E), lambda: ops.plan(idx, E, -1, 9), lambda: ops.plan(idx, 0),
                lambda: ops.swiglu_forward(xp[None], wg, wg, wd, p.offsets),
                lambda: ops.swiglu_backward(xp, xp, act, hgu, wg[0], wg, wd, p.offsets)):
        with pytest.raises(ValueError):
            bad()
    for bad in (lambda: ops.router_forward(x.half(), gw, K), lambda: ops.combine(y.double(), w, p),
                lambda: ops.unpermute_sum(y.half(), p), lambda: ops.swiglu_forward(xp.float(), wg, wg, wd, p.offsets)):
        with pytest.raises(TypeError):
            bad()
    with pytest.raises(RuntimeError, match="GPU"):
        ops.combine(y.cpu(), w, p)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_no_tokens(data, dtype):
    x, gw, nw = data(0, H, dtype=dtype), data(H, E, dtype=dtype), data(H, dtype=dtype)
    for out in (ops.router_forward(x, gw, K, aux_coef=0.01, z_coef=0.001, with_losses=True),
                ops.rmsnorm_router_forward(x, nw, 1e-6, gw, K, None, 0.01, 0.001)[2:]):
        idx, w, logits, lse, cnt, stats, aux, z = out
        assert idx.shape == w.shape == (0, K) and logits.shape == (0, E) and lse.shape == (0,)
        assert cnt.sum() == 0 and stats.abs().sum() == 0 and aux == 0 and z == 0
    p = ops.plan(idx, E, 3)
    assert p.rows == 0 and p.drop.shape == (0, K) and p.slot_row.numel() == 0 and int(p.ndrop) == 0
    assert int(p.offsets[-1]) == 0 and ops.permute(x, p).shape == (0, H)
