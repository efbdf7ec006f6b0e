"""Persistent solvers on assembled rows: rows with many entries, and the solvers
that contexts without memory for rows run instead.

Tolerances against the oracle: an FP64 CG to eps 1e-10 differs by rounding that
CG amplifies, 1e-10 of the solution; a mixed solve and the oracle stop at eps
1e-9, so their solutions agree within the condition number of the scaled system
(under 100 for these time steps) times that, 1e-7. GMRES: 2e-8 in FP64 (eps 1e-10
on both sides), 2e-7 mixed (eps 1e-9)."""
import ctypes

import numpy as np
import pytest
import torch

from opentelemac_amd import bief, mesh as M, system as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _fans(counts, rings=12):
    """Discs side by side, one per count: a centre with that many neighbours
    and rings of triangles around it."""
    xs, ys, tri, base = [], [], [], 0
    for d, s in enumerate(counts):
        a = 2.0 * np.pi * np.arange(s) / s
        r = np.arange(1, rings + 1)[:, None]
        xs.append(np.concatenate([[0.0], (r * np.cos(a)).ravel()]) + 2.5 * rings * d)
        ys.append(np.concatenate([[0.0], (r * np.sin(a)).ravel()]))
        i, j = np.arange(s), (np.arange(s) + 1) % s
        at = lambda q, k: base + 1 + q * s + k  # noqa: E731
        tri.append(np.stack([np.full(s, base), at(0, i), at(0, j)]))
        for q in range(rings - 1):
            tri.append(np.stack([at(q, i), at(q + 1, i), at(q + 1, j)]))
            tri.append(np.stack([at(q, i), at(q + 1, j), at(q, j)]))
        base += 1 + rings * s
    return M.Mesh(x=np.concatenate(xs), y=np.concatenate(ys),
                  ikle=np.concatenate(tri, axis=1).astype(np.int32))


@pytest.mark.parametrize("filler", [270000, 600000, 1100000])
def test_long_rows_give_the_same_bits_in_any_partition(gpu, filler):
    """Nodes of 9 to 40 neighbours: a row's terms are added in one order
    whether a workgroup holds 1 slab (alone) or, beside a large mesh, 2, 4 or 8."""
    fans = _fans(range(9, 41))
    meshes = [fans, M.channel_mesh_n(filler, seed=1, length=20.0 * filler ** 0.5,
                                     width=15.0 * filler ** 0.5)]
    systems = [S.wave_system(m, 2.0 + np.abs(m.x) / m.x.max(), dt=1.0) for m in meshes]
    for sd, m in zip(systems, meshes):
        sd["b"] = sd["b"] + 1e-2 * np.random.default_rng(5).normal(size=m.npoin)
    cat = lambda key: np.concatenate([s[key] for s in systems], axis=-1)  # noqa: E731
    ens = bief.Ensemble(meshes)
    ctx = bief.Context(fans)
    sd = systems[0]
    for prec in (bief.PREC_FP64, bief.PREC_MIXED):
        kw = dict(slv=1, precon=2, eps=1e-9, nitmax=500, precision=prec)
        ens.set_matrix("Q", "S", cat("da"), cat("xa"))
        x, _ = ens.solve(cat("x0"), cat("b"), **kw)
        ctx.set_matrix("Q", "S", sd["da"], sd["xa"])
        xa, ia = ctx.solve(sd["x0"].copy(), sd["b"].copy(), **kw)
        assert ia["converged"] and ens.infos()[0]["niter"] == ia["niter"]
        assert ens.infos()[0]["relres"] == ia["relres"]
        assert np.array_equal(ens.split(x)[0], xa)
    ctx.close()
    ens.close()


CG, GMRES = 1, 7
TOL = {(CG, bief.PREC_FP64): 1e-10, (CG, bief.PREC_MIXED): 1e-7,
       (GMRES, bief.PREC_FP64): 2e-8, (GMRES, bief.PREC_MIXED): 2e-7}


def _case(nx, ny, seed=3):
    m = M.random_small_mesh(nx, ny, seed=seed)
    sd = S.wave_system(m, 2.0 + m.x / 10.0, dt=0.3)
    sd["b"] = sd["b"] + 1e-2 * np.random.default_rng(seed).normal(size=m.npoin)
    return m, sd


def _against_oracle(ctx, m, sd, slv, prec, precon=2, typext="S"):
    """Two solves of the system (the second one launched as the first one's
    iterations have it planned)."""
    eps = 1e-10 if prec == bief.PREC_FP64 else 1e-9
    xa = sd["xa"] if typext == "S" else np.concatenate([sd["xa"], 0.5 * sd["xa"]])
    if slv == CG and typext == "Q":
        xa = np.concatenate([sd["xa"], sd["xa"]])
    kw = dict(slv=slv, precon=precon, eps=eps, nitmax=2000, krylov=6)
    xr, ir, _, _ = O.solve(O.Matrix(sd["da"], xa, "Q", typext), m.ikle, sd["b"], sd["x0"], **kw)
    for _ in range(2):
        ctx.set_matrix("Q", typext, sd["da"], xa)
        x, info = ctx.solve(sd["x0"].copy(), sd["b"].copy(), precision=prec, **kw)
        assert info["converged"], info
        if prec == bief.PREC_FP64:
            assert abs(info["niter"] - ir.niter) <= 1, (info, ir.niter)
        assert np.linalg.norm(x - xr) <= TOL[slv, prec] * np.linalg.norm(xr), info


@pytest.fixture
def no_rows(monkeypatch):
    monkeypatch.setenv("BHIP_ROWS_BYTES", "0")


@pytest.mark.parametrize("prec", [bief.PREC_FP64, bief.PREC_MIXED])
@pytest.mark.parametrize("slv", [CG, GMRES])
def test_solves_run_on_rows(gpu, slv, prec):
    m, sd = _case(70, 61)
    ctx = bief.Context(m)
    assert ctx.rows()["bytes"] > 0 and ctx.rows()["last_solve"] is None
    _against_oracle(ctx, m, sd, slv, prec)
    assert ctx.rows()["last_solve"] is True
    ctx.close()


@pytest.mark.parametrize("typext", ["S", "Q"])
@pytest.mark.parametrize("precon", [0, 2, 5])
@pytest.mark.parametrize("prec", [bief.PREC_FP64, bief.PREC_MIXED])
@pytest.mark.parametrize("slv", [CG, GMRES])
def test_solves_without_memory_for_rows(gpu, no_rows, slv, prec, precon, typext):
    """Element by element: the two-kernel CG and the GMRES driven from the host."""
    m, sd = _case(70, 61)
    ctx = bief.Context(m)
    assert ctx.rows()["bytes"] == 0
    _against_oracle(ctx, m, sd, slv, prec, precon, typext)
    assert ctx.rows()["last_solve"] is False
    ctx.close()


@pytest.mark.parametrize("prec", [bief.PREC_FP64, bief.PREC_MIXED])
def test_ensembles_without_memory_for_rows(gpu, no_rows, prec):
    cases = [_case(8 + 9 * k, 30 - 4 * k, seed=k) for k in range(5)]
    cases[2][1]["b"][:] = 0.0  # X = 0
    cat = lambda key: np.concatenate([s[key] for _, s in cases], axis=-1)  # noqa: E731
    eps = 1e-10 if prec == bief.PREC_FP64 else 1e-9
    kw = dict(slv=CG, precon=2, eps=eps, nitmax=500)
    ens = bief.Ensemble([m for m, _ in cases])
    for _ in range(2):
        ens.set_matrix("Q", "S", cat("da"), cat("xa"))
        x, info = ens.solve(cat("x0"), cat("b"), precision=prec, **kw)
        assert info["converged"] and ens.rows()["last_solve"] is False
        for (m, sd), xs, si in zip(cases, ens.split(x), ens.infos()):
            xr, ir, _, _ = O.solve(O.Matrix(sd["da"], sd["xa"], "Q", "S"), m.ikle, sd["b"],
                                   sd["x0"], **kw)
            assert np.linalg.norm(xs - xr) <= TOL[CG, prec] * np.linalg.norm(xr)
            if prec == bief.PREC_FP64:
                assert abs(si["niter"] - ir.niter) <= 1
    ens.close()


def test_static_scratch_without_memory_for_rows(gpu, no_rows):
    """The entry point without allocations uses its static partial sums and
    states here, a smaller system's after a larger one's."""
    for nx, ny in ((60, 40), (14, 9)):
        m, sd = _case(nx, ny)
        ctx = bief.Context(m, block_nodes=64)
        out = []
        for noalloc in (False, True):
            ctx.set_matrix("Q", "S", sd["da"], sd["xa"])
            x, b = (torch.tensor(sd[k], device="cuda") for k in ("x0", "b"))
            if noalloc:
                cfg, info = bief.SolverCfg(CG, 2, 5, 1000, 1e-10, bief.PREC_FP64, 1e-4, 0), \
                    bief.SolveInfo()
                ctx._sync_torch()
                rc = bief.lib().bhip_solve_dev_noalloc(ctx._h, ctypes.byref(cfg), x.data_ptr(),
                                                       b.data_ptr(), ctypes.byref(info))
                torch.cuda.synchronize()
                assert rc == 0 and info.converged
            else:
                ctx.solve(x, b, slv=CG, precon=2, eps=1e-10, nitmax=1000)
            assert ctx.rows()["last_solve"] is False
            out.append((x, b))
        assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
        ctx.close()


def test_memory_that_runs_out_after_the_set_up(gpu, monkeypatch):
    """Enough for the FP64 rows, not for the FP32 ones nor for a basis: those
    solves run element by element, the others on rows."""
    m, sd = _case(70, 61)
    ctx = bief.Context(m)
    enough = ctx.rows()["bytes"]
    ctx.close()
    for limit, rows in ((enough, True), (enough - 1, False)):
        monkeypatch.setenv("BHIP_ROWS_BYTES", str(limit))
        ctx = bief.Context(m)
        assert ctx.rows()["bytes"] == (enough if rows else 0)
        for slv, prec, on in ((CG, bief.PREC_MIXED, False), (GMRES, bief.PREC_FP64, False),
                              (GMRES, bief.PREC_MIXED, False), (CG, bief.PREC_FP64, rows)):
            _against_oracle(ctx, m, sd, slv, prec)
            assert ctx.rows()["last_solve"] is on, (slv, prec, limit)
            assert ctx.rows()["bytes"] == (enough if rows else 0)
        ctx.close()


@pytest.mark.parametrize("slv", [CG, GMRES])
@pytest.mark.parametrize("prec", [bief.PREC_FP64, bief.PREC_MIXED])
def test_rows_are_tried_again_after_a_launch_gave_up(gpu, monkeypatch, capfd, slv, prec):
    """The solve that a launch gave up and the next 64 run element by element, with
    one line about it; then the rows serve again, to the same bits as ever."""
    m, sd = _case(70, 61)
    eps = 1e-10 if prec == bief.PREC_FP64 else 1e-9

    def solve(ctx):
        ctx.set_matrix("Q", "S", sd["da"], sd["xa"])
        x, info = ctx.solve(sd["x0"].copy(), sd["b"].copy(), slv=slv, precon=2, eps=eps,
                            nitmax=2000, krylov=6, precision=prec)
        assert info["converged"]
        return x, info["niter"], ctx.rows()["last_solve"]

    ctx = bief.Context(m)
    want = solve(ctx)
    assert want[2] is True
    ctx.close()
    monkeypatch.setenv("BHIP_ROWS_WAIT", "0")
    ctx = bief.Context(m)
    capfd.readouterr()
    first = solve(ctx)
    assert first[2] is False
    assert np.linalg.norm(first[0] - want[0]) <= TOL[slv, prec] * np.linalg.norm(want[0])
    assert capfd.readouterr().err.count("the next 64 solves") == 1
    for _ in range(64):
        assert solve(ctx)[2] is False
    monkeypatch.delenv("BHIP_ROWS_WAIT")
    for _ in range(3):
        x, niter, on = solve(ctx)
        assert on is True and niter == want[1] and np.array_equal(x, want[0])
    assert "solves" not in capfd.readouterr().err
    ctx.close()


@pytest.mark.parametrize("prec", [bief.PREC_FP64, bief.PREC_MIXED])
def test_latencies_count_from_the_start_of_the_solve(gpu, prec):
    """1024 equal systems on 256 CUs, a workgroup each: the ones that wait for a CU
    are told by their latencies. A zero right-hand side takes no time."""
    m, sd = _case(29, 31)
    n = 1024
    ens = bief.Ensemble([m] * n)
    rep = lambda a: np.concatenate([a] * n, axis=-1)  # noqa: E731
    b = np.tile(sd["b"], (n, 1))
    b[5] = 0.0
    ens.set_matrix("Q", "S", rep(sd["da"]), rep(sd["xa"]))
    _, info = ens.solve(rep(sd["x0"]), b.ravel(), slv=CG, precon=2, eps=1e-9, nitmax=500,
                        precision=prec)
    assert info["converged"] and ens.rows()["last_solve"] is True
    ms = np.array(ens.latencies_ms())
    assert ms[5] == 0.0
    ms = np.delete(ms, 5)
    assert ms.min() > 0.0 and ms.max() >= 2.0 * ms.min()
    ens.close()


def test_wide_systems_beyond_the_gpu(gpu):
    """Ten systems of 37 workgroups of 8 slabs each: more than the GPU holds, and
    each wider than an XCD. Whole systems per launch; the bits of each alone."""
    m = M.channel_mesh(600, 498, 12000.0, 9960.0)
    sd = S.wave_system(m, 2.0 + m.x / m.x.max(), dt=1.0)
    rng = np.random.default_rng(3)
    n = 10
    b = sd["b"] + 1e-2 * rng.normal(size=(n, m.npoin))
    rep = lambda a: np.concatenate([a] * n, axis=-1)  # noqa: E731
    ens, one = bief.Ensemble([m] * n), bief.Context(m)
    for prec in (bief.PREC_FP64, bief.PREC_MIXED):
        kw = dict(slv=CG, precon=2, eps=1e-9, nitmax=500, precision=prec)
        ens.set_matrix("Q", "S", rep(sd["da"]), rep(sd["xa"]))
        x, info = ens.solve(rep(sd["x0"]), b.flatten(), **kw)
        assert info["converged"] and ens.rows()["last_solve"] is True
        ms = np.array(ens.latencies_ms())
        assert ms.min() > 0.0 and ms[-1] > ms[0]
        for k in (0, 5, 6, 9):
            one.set_matrix("Q", "S", sd["da"], sd["xa"])
            xa, ia = one.solve(sd["x0"].copy(), b[k].copy(), **kw)
            assert one.rows()["last_solve"] is True and ens.infos()[k]["niter"] == ia["niter"]
            assert np.array_equal(ens.split(x)[k], xa)
    ens.close()
    one.close()
