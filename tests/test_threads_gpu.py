"""Router forwards from several host threads on one stream: the calls share the stream's workspace, through which the
launches of one call hand data on (the packed gate, the per-block partials), so no other call's launches may come
between them.  Every result has the bits of the same call made alone."""

from __future__ import annotations

import threading

import pytest
import torch

from gpu_util import dev, say

from moe_mi355 import ops
from moe_mi355.router import route

pytestmark = pytest.mark.gpu

B, F = torch.bfloat16, torch.float32
# (E, H, dtype of x, dtype of the gate): packed gate (few-token form), E <= 32 streaming (one launch), the general
# kernels (a gate of another type), fp32
FORMS = [(64, 256, B, B), (128, 256, B, B), (8, 256, B, B), (24, 200, B, F), (64, 128, F, F)]


def _calls(E, H, xd, gd, seed):
    """Three entry points that take the stream's workspace, as functions of no argument."""
    g = torch.Generator().manual_seed(seed)
    n = 48 + 16 * (seed % 3)
    x = torch.randn(n, H, generator=g).to(xd).to(dev())
    w = (torch.randn(H, E, generator=g) * H**-0.5).to(gd).to(dev())
    nw = torch.ones(H, device=dev())
    return [
        lambda: ops.router_forward(x, w, 4, aux_coef=0.01, z_coef=1e-3, with_losses=True),
        lambda: ops.rmsnorm_router_forward(x, nw, 1e-5, w, 4, aux_coef=0.01, z_coef=1e-3),
        lambda: route(x.detach().requires_grad_(True), w, 4, 0.01, 1e-3),
    ]


@pytest.mark.parametrize("form", FORMS, ids=lambda f: f"E{f[0]}-H{f[1]}-{str(f[2])[6:]}-{str(f[3])[6:]}")
def test_threads_on_one_stream(form):
    say(f"[threads] {form}")
    T, rounds = 4, 40
    calls = [_calls(*form, seed=i) for i in range(T)]
    alone = [[[t.detach().clone() for t in f()] for f in fs] for fs in calls]
    torch.cuda.synchronize()
    got, errors = [[] for _ in range(T)], []
    start = threading.Barrier(T)

    def work(i):
        try:
            start.wait(30)
            for r in range(rounds):
                for j in range(3):
                    k = (i + j + r) % 3
                    got[i].append((k, [t.detach() for t in calls[i][k]()]))
        except Exception as e:  # re-raised by the test's own thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(T)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for i in range(T):
        assert len(got[i]) == 3 * rounds
        for k, outs in got[i]:
            for a, b in zip(outs, alone[i][k]):
                assert torch.equal(a, b)
