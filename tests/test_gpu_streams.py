"""Ordering between the context's stream and the caller's: results that the
caller's stream reads at once, inputs it has only queued, from side streams and
from two threads with a context each."""
import threading

import numpy as np
import pytest
import torch

from opentelemac_amd import bief, mesh as M, system as S, tracer

pytestmark = pytest.mark.gpu


def _case(seed):
    m = M.random_small_mesh(120, 90, seed=seed)
    sd = S.wave_system(m, 2.0 + m.x / 10.0, dt=0.3)
    ctx = bief.Context(m)
    ctx.set_matrix("Q", "S", sd["da"], sd["xa"])
    return m, ctx


def _chain(ctx, y, steps=20):
    """Products whose inputs and outputs pass through queued work of torch."""
    scale = torch.ones(1, dtype=torch.float64, device="cuda")
    for _ in range(200):
        scale = scale * 1.0  # a queue in front of the first product
    v = y * scale
    for _ in range(steps):
        v = ctx.matvec("X=AY", v)
        v = v / v.abs().max()
    return v


@pytest.mark.parametrize("side", [False, True])
def test_products_and_torch_work_alternate(gpu, side):
    m, ctx = _case(1)
    y = torch.rand(m.npoin, dtype=torch.float64, device="cuda")
    with torch.cuda.stream(ctx.torch_stream()):
        want = _chain(ctx, y)
    torch.cuda.synchronize()
    s = torch.cuda.Stream() if side else torch.cuda.current_stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = _chain(ctx, y)
        same = torch.equal(got, want)
    assert same
    ctx.close()


def test_two_threads(gpu):
    cases = [_case(k) for k in (2, 3)]
    ys = [torch.rand(m.npoin, dtype=torch.float64, device="cuda") for m, _ in cases]
    want = []
    for (_, ctx), y in zip(cases, ys):
        with torch.cuda.stream(ctx.torch_stream()):
            want.append(_chain(ctx, y))
        torch.cuda.synchronize()
    ok = [False, False]

    def run(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            ok[k] = all(torch.equal(_chain(cases[k][1], ys[k]), want[k]) for _ in range(5))

    ts = [threading.Thread(target=run, args=(k,)) for k in (0, 1)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert ok == [True, True]
    for _, ctx in cases:
        ctx.close()


def test_supg_system_is_ordered_with_the_caller(gpu):
    """The right-hand side follows a velocity that is still being computed, and
    is what host arrays give."""
    m = M.channel_mesh(60, 40, 6000.0, 2400.0)
    u, v, fn, _ = tracer.estuary_flow(m, seed=3)
    nu = np.full(m.npoin, 0.1)
    host = bief.Context(m)
    want = tracer.supg_system(host, m, u, v, nu, 10.0, fn, tetat=0.6)
    ctx = bief.Context(m)
    dev = lambda a: torch.tensor(a, device="cuda")  # noqa: E731
    du, dv, dn, df = dev(u), dev(v), dev(nu), dev(fn)
    tracer.supg_system(ctx, m, du, dv, dn, 10.0, df, tetat=0.6)
    for _ in range(3):
        t = du * 0.0
        for _ in range(100):
            t = t + du / 100.0
        sm = tracer.supg_system(ctx, m, t * 1.0, dv, dn, 10.0, df, tetat=0.6)
        got = (sm * 1.0).cpu().numpy()
        # t is u to 100 roundings
        assert np.abs(got - want).max() <= 1e-12 * np.abs(want).max()
    host.close()
    ctx.close()


@pytest.mark.parametrize("shift", [0, 1])
def test_product_onto_its_operand(gpu, shift):
    """x is y, or overlaps it: the same bits as with vectors of their own."""
    m, ctx = _case(4)
    n = m.npoin
    buf = torch.rand(n + 1, dtype=torch.float64, device="cuda")
    for op in bief.OPS:
        b = buf.clone()
        y, x = b[:n], b[shift:shift + n]
        want = ctx.matvec(op, y.clone(), x.clone(), c=0.75)
        got = ctx.matvec(op, y, x, c=0.75)
        assert torch.equal(got, want), op
    ctx.close()
