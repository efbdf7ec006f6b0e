"""Element matrices summed onto the nodes of a block, a window of slots at a
time: blocks of one window and of several, more and fewer than 256 of them
(the workgroup's size changes there), against sums in numpy.

Tolerance: a node sums at most some 12 terms whose factors differ from
numpy's by a few roundings, 1e-13 of the largest diagonal term."""
import numpy as np
import pytest
import torch

from opentelemac_amd import bief, mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block_nodes", [37, 64, 300, 1024, 3000])
def test_diagonals_over_windows_of_slots(gpu, block_nodes):
    m = M.channel_mesh_n(17000, seed=2, length=1700.0, width=1000.0)
    xe, ye = m.x[m.ikle], m.y[m.ikle]
    x2, x3 = xe[1] - xe[0], xe[2] - xe[0]
    y2, y3 = ye[1] - ye[0], ye[2] - ye[0]
    s = 0.5 * (x2 * y3 - x3 * y2)
    zero = np.zeros_like(x2)
    rng = np.random.default_rng(block_nodes)
    u, v = rng.uniform(0.5, 1.5, m.npoin), rng.uniform(0.5, 1.5, m.npoin)
    ctx = bief.Context(m, block_nodes=block_nodes)
    ctx.set_geometry(np.stack([zero, x2, x3]), np.stack([zero, y2, y3]), s)

    def check(terms, what):
        want = np.zeros(m.npoin)
        for k in range(3):
            np.add.at(want, m.ikle[k], terms[k])
        _, da, _ = ctx.get_matrix()
        assert np.abs(da - want).max() <= 1e-13 * np.abs(want).max(), what

    ctx.matrix_mt01aa(3.0, None)
    mass = [s * (3.0 / 6.0)] * 3
    check(mass, "mass")
    dev = lambda a: torch.tensor(a, device="cuda")  # noqa: E731
    ctx.matrix_mt02aa(1, 2.0, None, None, None, dev(u), accumulate=True)
    som = u[m.ikle].sum(axis=0) * (2.0 / 12.0) / s
    a12 = -som * (x3 * (x3 - x2) + y3 * (y3 - y2))
    a13 = som * (x2 * (x3 - x2) + y2 * (y3 - y2))
    a23 = -som * (x2 * x3 + y2 * y3)
    both = [mass[0] - a12 - a13, mass[1] - a12 - a23, mass[2] - a13 - a23]
    check(both, "mass + diffusion")
    # MT04AA: (U.grad phi_i)(U.grad phi_i), the mean of U.grad^2 over the
    # element by the mid-edge rule (exact for quadratics)
    ctx.matrix_supg(4, 1.0, None, None, None, dev(u), dev(v))
    gx = np.stack([y2 - y3, y3, -y2]) / (2 * s)
    gy = np.stack([x3 - x2, -x3, x2]) / (2 * s)
    ue, ve = u[m.ikle], v[m.ikle]
    terms = []
    for i in range(3):
        q = [((ue[a] + ue[b]) / 2 * gx[i] + (ve[a] + ve[b]) / 2 * gy[i]) ** 2
             for a, b in ((0, 1), (1, 2), (2, 0))]
        terms.append(s * sum(q) / 3.0)
    check(terms, "MT04AA")
    ctx.close()
