"""CG and GMRES on assembled rows (one persistent launch per solve): the sizes where its
partition changes, against the oracle, and the path it falls back to.

Tolerances: FP64 solves to eps 1e-10 differ from the oracle's by rounding that
CG amplifies, 1e-10 of the solution as in the other solve tests; a mixed solve
and the oracle both stop at a relative residual of eps 1e-9, so their
solutions agree within the condition number of the scaled system (under 100
for these time steps) times that, 1e-7. GMRES likewise: 2e-8 in FP64 (eps 1e-10
on both sides), 2e-7 mixed (eps 1e-9)."""
import numpy as np
import pytest
import torch

from opentelemac_amd import bief, mesh as M, system as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _system(m):
    return S.wave_system(m, 2.0 + m.x / m.x.max(), dt=1.0)


def _check(m, sysd, precon=2, block_nodes=0, typext="S", seed=0):
    rng = np.random.default_rng(seed)
    b = sysd["b"] + 1e-2 * rng.normal(size=m.npoin)
    xa = sysd["xa"] if typext == "S" else np.concatenate([sysd["xa"], sysd["xa"]])
    A = O.Matrix(sysd["da"], xa, "Q", typext)
    out = []
    for prec, eps, tol in ((bief.PREC_FP64, 1e-10, 1e-10), (bief.PREC_MIXED, 1e-9, 1e-7)):
        xr, ir, _, _ = O.solve(A, m.ikle, b, sysd["x0"], slv=1, precon=precon, eps=eps,
                               nitmax=2000)
        ctx = bief.Context(m, block_nodes=block_nodes)
        ctx.set_matrix("Q", typext, sysd["da"], xa)
        x, info = ctx.solve(sysd["x0"].copy(), b.copy(), slv=1, precon=precon, eps=eps,
                            nitmax=2000, precision=prec)
        assert info["converged"], info
        if prec == bief.PREC_FP64:
            assert abs(info["niter"] - ir.niter) <= 1, (info, ir.niter)
        assert np.linalg.norm(x - xr) <= tol * np.linalg.norm(xr), (prec, info)
        out.append(x)
        ctx.close()
    return out


# nodes around one slab of 1024 rows, and the first sizes of 2, 4 and 8 slabs
# per workgroup
@pytest.mark.parametrize("nx,ny", [(1, 1), (30, 32), (31, 31), (24, 40), (682, 2), (514, 510),
                                   (730, 719), (1030, 1020)])
def test_rows_cg_at_partition_edges(gpu, nx, ny):
    m = M.channel_mesh(nx, ny, 10.0 * nx, 10.0 * ny)
    _check(m, _system(m))


@pytest.mark.parametrize("precon", [0, 5])
@pytest.mark.parametrize("typext", ["S", "Q"])
def test_rows_cg_with_a_diagonal(gpu, precon, typext):
    """No unit diagonal (PRECON 5, none) and coefficients stored in both
    halves; node blocks that do not match the slabs."""
    m = M.random_small_mesh(70, 61, seed=3)
    _check(m, S.wave_system(m, 2.0 + m.x / 10.0, dt=0.3), precon=precon, block_nodes=300,
           typext=typext)


@pytest.mark.parametrize("precon", [0, 2, 5])
@pytest.mark.parametrize("typext", ["S", "Q"])
def test_rows_summed_with_the_scaling(gpu, precon, typext):
    """Node blocks that are the slabs (1024 rows, the last one ragged): rows
    summed in the pass that scales the coefficients, or that only reads them;
    from the context's matrix and from the saved copy."""
    m = M.random_small_mesh(70, 61, seed=4)
    sysd = S.wave_system(m, 2.0 + m.x / 10.0, dt=0.3)
    want = _check(m, sysd, precon=precon, block_nodes=1024, typext=typext)[0]
    rng = np.random.default_rng(0)
    b = sysd["b"] + 1e-2 * rng.normal(size=m.npoin)
    ctx = bief.Context(m, block_nodes=1024)
    xa = sysd["xa"] if typext == "S" else np.concatenate([sysd["xa"], sysd["xa"]])
    ctx.set_matrix("Q", typext, sysd["da"], xa)
    ctx.save_matrix()
    for _ in range(2):
        dx, db = torch.tensor(sysd["x0"], device="cuda"), torch.tensor(b, device="cuda")
        ctx.solve(dx, db, slv=1, precon=precon, eps=1e-10, nitmax=2000, restore=True)
        assert np.array_equal(dx.cpu().numpy(), want)
    ctx.close()


def test_rows_of_a_diagonal_matrix(gpu):
    """No off-diagonal terms (TYPEXT '0'): the rows hold zeros."""
    m = M.random_small_mesh(40, 31, seed=5)
    sysd = S.wave_system(m, 2.0 + m.x / 10.0, dt=0.3)
    ctx = bief.Context(m, block_nodes=1024)
    ctx.set_matrix("Q", "S", sysd["da"], sysd["xa"])
    ctx.solve(sysd["x0"].copy(), sysd["b"].copy(), slv=1, precon=2, eps=1e-8, nitmax=100)
    for precon in (0, 2):
        ctx.set_matrix("Q", "0", sysd["da"], None)
        x, info = ctx.solve(sysd["x0"].copy(), sysd["b"].copy(), slv=1, precon=precon, eps=1e-12,
                            nitmax=4000)
        assert info["converged"]
        np.testing.assert_allclose(x, sysd["b"] / sysd["da"],
                                   atol=1e-10 * np.abs(sysd["b"] / sysd["da"]).max())
    ctx.close()


@pytest.mark.parametrize("nx,ny", [(20, 12), (120, 90), (514, 510)])
@pytest.mark.parametrize("precon", [0, 2])
def test_rows_cg_from_an_initial_solution(gpu, nx, ny, precon):
    """R = A X0 - B and its exchange inside the launch; a solve that NITMAX ends,
    one that X0 ends, and a zero right-hand side."""
    m = M.channel_mesh(nx, ny, 10.0 * nx, 10.0 * ny)
    sysd = _system(m)
    rng = np.random.default_rng(7)
    x0 = rng.normal(size=m.npoin)
    b = sysd["b"] + 1e-2 * rng.normal(size=m.npoin)
    A = O.Matrix(sysd["da"], sysd["xa"], "Q", "S")

    def both(x0, b, **kw):
        kw = dict(dict(slv=1, precon=precon, eps=1e-10, nitmax=3000), **kw)
        xr, ir, br, _ = O.solve(A, m.ikle, b, x0, **kw)
        ctx = bief.Context(m)
        ctx.set_matrix("Q", "S", sysd["da"], sysd["xa"])
        bh = b.copy()
        x, info = ctx.solve(x0.copy(), bh, **kw)
        ctx.close()
        assert bool(info["converged"]) == bool(ir.converged)
        return x, xr, info, ir

    x, xr, info, ir = both(x0, b)
    assert abs(info["niter"] - ir.niter) <= 1
    assert np.linalg.norm(x - xr) <= 1e-10 * np.linalg.norm(xr)
    # few iterations: no rounding has grown yet
    x, xr, info, ir = both(x0, b, nitmax=3)
    assert info["niter"] == ir.niter == 3
    assert np.linalg.norm(x - xr) <= 1e-12 * np.linalg.norm(xr)
    x, _, info, _ = both(xr, b, eps=1e30)
    assert info["niter"] == 0
    np.testing.assert_allclose(x, xr, rtol=1e-15)
    x, _, info, _ = both(x0, np.zeros(m.npoin))
    assert info["niter"] == 0 and not x.any()


def test_more_workgroups_than_the_gpu_holds(gpu):
    """300 systems of one workgroup each: workgroups numbered as they start."""
    meshes = [M.random_small_mesh(4 + k % 5, 5 + k % 3, seed=k) for k in range(300)]
    systems = [S.wave_system(m, 2.0 + m.x / 10.0, dt=1.0 + 0.01 * k)
               for k, m in enumerate(meshes)]
    cat = lambda key: np.concatenate([s[key] for s in systems], axis=-1)  # noqa: E731
    ens = bief.Ensemble(meshes)
    for prec, eps, tol in ((bief.PREC_FP64, 1e-10, 1e-10), (bief.PREC_MIXED, 1e-9, 1e-7)):
        ens.set_matrix("Q", "S", cat("da"), cat("xa"))
        x, info = ens.solve(cat("x0"), cat("b"), slv=1, precon=2, eps=eps, nitmax=500,
                            precision=prec)
        assert info["converged"]
        for m, sd, xs, si in zip(meshes, systems, ens.split(x), ens.infos()):
            xr, ir, _, _ = O.solve(O.Matrix(sd["da"], sd["xa"], "Q", "S"), m.ikle, sd["b"],
                                   sd["x0"], slv=1, precon=2, eps=eps, nitmax=500)
            assert np.linalg.norm(xs - xr) <= tol * np.linalg.norm(xr)
            if prec == bief.PREC_FP64:
                assert abs(si["niter"] - ir.niter) <= 1


@pytest.mark.parametrize("filler", [270000, 600000, 1100000])
def test_a_member_gives_the_same_bits_in_any_partition(gpu, filler):
    """Sums are trees over rows: a system solved alone (one slab per
    workgroup) and beside a mesh that makes the context use 2, 4 or 8."""
    meshes = [M.channel_mesh_n(n, seed=k, length=20.0 * n ** 0.5, width=15.0 * n ** 0.5)
              for k, n in enumerate((2500, 21000, filler))]
    systems = [S.wave_system(m, 2.0 + m.x / m.x.max(), dt=1.0) for m in meshes]
    cat = lambda key: np.concatenate([s[key] for s in systems], axis=-1)  # noqa: E731
    ens = bief.Ensemble(meshes)
    for prec in (bief.PREC_FP64, bief.PREC_MIXED):
        kw = dict(slv=1, precon=2, eps=1e-9, nitmax=500, precision=prec)
        ens.set_matrix("Q", "S", cat("da"), cat("xa"))
        x, _ = ens.solve(cat("x0"), cat("b"), **kw)
        for m, sd, xs, si in zip(meshes[:2], systems, ens.split(x), ens.infos()):
            ctx = bief.Context(m)
            ctx.set_matrix("Q", "S", sd["da"], sd["xa"])
            xa, ia = ctx.solve(sd["x0"].copy(), sd["b"].copy(), **kw)
            assert si["niter"] == ia["niter"] and si["relres"] == ia["relres"]
            assert np.array_equal(xs, xa)
            ctx.close()
    ens.close()


def test_a_launch_that_gives_up_falls_back(gpu, monkeypatch):
    """A limit of zero on the workgroups' waits: the persistent launch gives up
    at its first meeting and the two-kernel CG solves the system."""
    m = M.channel_mesh(120, 90, 1200.0, 900.0)
    sysd = _system(m)
    want = _check(m, sysd)
    monkeypatch.setenv("BHIP_ROWS_WAIT", "0")
    got = _check(m, sysd)
    assert np.linalg.norm(got[0] - want[0]) <= 1e-10 * np.linalg.norm(want[0])


def _check_gmres(m, sysd, krylov, precon=2, typext="S", block_nodes=0, seed=1):
    rng = np.random.default_rng(seed)
    b = sysd["b"] + 1e-2 * rng.normal(size=m.npoin)
    xa = sysd["xa"]
    if typext == "Q":
        # not symmetric, still diagonally dominant
        xa = np.concatenate([sysd["xa"], 0.5 * sysd["xa"]])
    A = O.Matrix(sysd["da"], None if typext == "0" else xa, "Q", typext)
    for prec, eps, tol in ((bief.PREC_FP64, 1e-10, 2e-8), (bief.PREC_MIXED, 1e-9, 2e-7)):
        if krylov == 1:
            # the oracle's residual estimate ||A V||^2 - H^2 loses all its
            # digits below 1e-9 here (its relres is then 0)
            eps, tol = 1e-8, 2e-6
        kw = dict(slv=7, precon=precon, eps=eps, nitmax=400, krylov=krylov)
        xr, ir, _, _ = O.solve(A, m.ikle, b, sysd["x0"], **kw)
        ctx = bief.Context(m, block_nodes=block_nodes)
        ctx.set_matrix("Q", typext, sysd["da"], None if typext == "0" else xa)
        x, info = ctx.solve(sysd["x0"].copy(), b.copy(), precision=prec, **kw)
        assert info["converged"], (prec, info)
        if prec == bief.PREC_FP64:
            assert abs(info["niter"] - ir.niter) <= 1, (info, ir.niter)
        assert np.linalg.norm(x - xr) <= tol * np.linalg.norm(xr), (prec, info)
        ctx.close()


# one workgroup; several; 2, 4 and 8 slabs each
@pytest.mark.parametrize("nx,ny,krylov", [(1, 1, 2), (30, 32, 5), (120, 90, 1), (120, 90, 2),
                                          (120, 90, 20), (514, 510, 5), (730, 719, 3),
                                          (1030, 1020, 3)])
def test_rows_gmres_at_partition_edges(gpu, nx, ny, krylov):
    m = M.channel_mesh(nx, ny, 10.0 * nx, 10.0 * ny)
    _check_gmres(m, _system(m), krylov)


@pytest.mark.parametrize("block_nodes", [300, 1024])
@pytest.mark.parametrize("precon", [0, 2, 5])
@pytest.mark.parametrize("typext", ["S", "Q"])
def test_rows_gmres_with_a_diagonal(gpu, precon, typext, block_nodes):
    m = M.random_small_mesh(70, 61, seed=3)
    _check_gmres(m, S.wave_system(m, 2.0 + m.x / 10.0, dt=0.3), 6, precon=precon, typext=typext,
                 block_nodes=block_nodes)


def test_rows_gmres_reduces_the_krylov_space(gpu):
    """The unit matrix and a right-hand side whose norm is a power of two: A V_1
    is V_1 to the bit, so the cycle stops at one vector."""
    m = M.random_small_mesh(40, 31, seed=5)
    b = np.zeros(m.npoin)
    b[[3, 400, 800, 1200]] = 8.0
    for prec in (bief.PREC_FP64, bief.PREC_MIXED):
        ctx = bief.Context(m)
        ctx.set_matrix("Q", "0", np.ones(m.npoin), None)
        x, info = ctx.solve(np.zeros(m.npoin), b.copy(), slv=7, precon=0, eps=1e-10, nitmax=9,
                            krylov=4, precision=prec)
        assert info["converged"] and info["niter"] == 1 and info["relres"] == 0.0, info
        assert np.array_equal(x, b)
        ctx.close()


def test_a_gmres_launch_that_gives_up_falls_back(gpu, monkeypatch):
    monkeypatch.setenv("BHIP_ROWS_WAIT", "0")
    m = M.channel_mesh(120, 90, 1200.0, 900.0)
    _check_gmres(m, _system(m), 5)


def test_mixed_gmres_of_residuals_beyond_float(gpu):
    """A right-hand side of 2^130 times another's: all operations scale by a
    power of two, so only FP32's range could tell the two apart. (1e-6: the
    scaled residual rounds elsewhere in FP32, both solves stop at 1e-9.)"""
    m = M.channel_mesh(120, 90, 1200.0, 900.0)
    sysd = _system(m)
    b = 1.0 + np.random.default_rng(3).random(m.npoin)
    out = []
    for scale in (1.0, 2.0 ** 130):
        ctx = bief.Context(m)
        ctx.set_matrix("Q", "S", sysd["da"], sysd["xa"])
        x, info = ctx.solve(np.zeros(m.npoin), b * scale, slv=7, precon=2, eps=1e-9, nitmax=100,
                            krylov=5, precision=bief.PREC_MIXED)
        assert info["converged"], info
        out.append(x / scale)
        ctx.close()
    assert np.linalg.norm(out[1] - out[0]) <= 1e-6 * np.linalg.norm(out[0])
