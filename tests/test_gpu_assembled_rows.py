"""Persistent solvers on assembled rows: rows with many entries."""
import numpy as np
import pytest

from opentelemac_amd import bief, mesh as M, system as S

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
