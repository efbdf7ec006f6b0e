"""Contexts made and destroyed in turn: large host arrays pass through a pinned
ring that outlives them all, and whose copies ran on their streams."""
import numpy as np
import pytest

from opentelemac_amd import bief, mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("overlap", [0, 1])
def test_large_host_copies_over_contexts(gpu, overlap):
    """Each context leaves the ring at another of its places (17 and 5 MB, chunks
    of 8); overlap: it is destroyed after the next one's copies."""
    meshes = [M.channel_mesh(600, 590, 6000.0, 5900.0), M.channel_mesh(400, 300, 4000.0, 3000.0)]
    rng = np.random.default_rng(1)
    alive = []
    for k in range(8):
        m = meshes[k % 2]
        da, xa = rng.normal(size=m.npoin), rng.normal(size=(3, m.nelem))
        ctx = bief.Context(m)
        ctx.set_matrix("Q", "S", da, xa)
        typdia, da2, xa2 = ctx.get_matrix()
        assert typdia == "Q" and np.array_equal(da2, da) and np.array_equal(xa2, xa)
        y = rng.normal(size=m.npoin)
        x = ctx.matvec("X=AY", y)
        i, j, k3 = m.ikle
        want = da * y
        for p, q, c in ((i, j, xa[0]), (i, k3, xa[1]), (j, k3, xa[2])):
            want += np.bincount(p, c * y[q], minlength=m.npoin)
            want += np.bincount(q, c * y[p], minlength=m.npoin)
        # a dozen terms of order 1 per node
        assert np.abs(x - want).max() <= 1e-13 * np.abs(want).max()
        alive.append(ctx)
        if len(alive) > overlap:
            alive.pop(0).close()
    for ctx in alive:
        ctx.close()
