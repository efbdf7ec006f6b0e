"""Solves of several processes and threads on one GPU."""
import fcntl
import glob
import os
import subprocess
import sys
import threading
import time

import numpy as np
import pytest

from opentelemac_amd import bief, mesh as M, system as S

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = r"""
import sys
import numpy as np
from opentelemac_amd import bief, mesh as M, system as S
m = M.channel_mesh(720, 690, 14400.0, 13800.0)
sd = S.wave_system(m, 2.0 + m.x / m.x.max(), dt=1.0)
ctx = bief.Context(m)
out = []
def solve(slv, prec):
    ctx.set_matrix("Q", "S", sd["da"], sd["xa"])
    x, info = ctx.solve(sd["x0"].copy(), sd["b"].copy(), slv=slv, precon=2, eps=1e-9, nitmax=500,
                        krylov=5, precision=prec)
    assert info["converged"] and ctx.rows()["last_solve"] is True, ctx.rows()
    return x
kinds = [(1, bief.PREC_FP64), (1, bief.PREC_MIXED), (7, bief.PREC_FP64)]
want = [solve(*k) for k in kinds]
print("ready", flush=True)
sys.stdin.readline()
for _ in range(30):
    for k, w in zip(kinds, want):
        assert np.array_equal(solve(*k), w), k
print("done", flush=True)
"""


def test_processes_take_turns(gpu):
    """Three processes with a system of 245 workgroups each: every solve runs on
    rows, to the same bits, and none complains."""
    ps = [subprocess.Popen([sys.executable, "-c", CHILD], cwd=ROOT, text=True,
                           stdin=subprocess.PIPE, stdout=subprocess.PIPE, stderr=subprocess.PIPE)
          for _ in range(3)]
    try:
        for p in ps:
            assert p.stdout.readline() == "ready\n", p.stderr.read()
        for p in ps:
            p.stdin.write("go\n")
            p.stdin.flush()
        for p in ps:
            out, err = p.communicate(timeout=90)
            assert out == "done\n" and p.returncode == 0 and "libbiefhip" not in err, err
    finally:
        for p in ps:
            if p.poll() is None:
                p.kill()


def _context(nx, ny):
    m = M.random_small_mesh(nx, ny, seed=3)
    sd = S.wave_system(m, 2.0 + m.x / 10.0, dt=0.3)
    ctx = bief.Context(m)

    def solve(slv=1, prec=bief.PREC_FP64):
        ctx.set_matrix("Q", "S", sd["da"], sd["xa"])
        x, info = ctx.solve(sd["x0"].copy(), sd["b"].copy(), slv=slv, precon=2, eps=1e-10,
                            nitmax=500, krylov=5, precision=prec)
        assert info["converged"]
        return x, ctx.rows()["last_solve"]
    return ctx, solve


@pytest.mark.parametrize("slv", [1, 7])
def test_a_gpu_that_another_process_keeps(gpu, capfd, slv):
    """While its file is locked elsewhere, a solve waits its time and runs element
    by element, and so do the next 64, at once and with one line about it; a system
    of one workgroup needs no turn. Then the rows serve again."""
    ctx, solve = _context(70, 61)
    one, solve_one = _context(20, 21)
    want = solve(slv)
    assert want[1] is True
    held = []
    for path in glob.glob("/dev/shm/bhip-gpu-*") + glob.glob("/tmp/bhip-gpu-*"):
        fd = os.open(path, os.O_RDONLY)
        fcntl.flock(fd, fcntl.LOCK_EX | fcntl.LOCK_NB)
        held.append(fd)
    assert held
    capfd.readouterr()
    t = time.perf_counter()
    for _ in range(65):
        x, on = solve(slv)
        assert on is False
        # both stop at eps 1e-10; the scaled system's condition number is below 100
        assert np.linalg.norm(x - want[0]) <= 2e-8 * np.linalg.norm(want[0])
    assert 2.0 <= time.perf_counter() - t <= 4.0
    assert capfd.readouterr().err.count("another process") == 1
    assert solve_one()[1] is True
    for fd in held:
        os.close(fd)
    x, on = solve(slv)
    assert on is True and np.array_equal(x, want[0])
    ctx.close()
    one.close()


def test_threads_with_a_context_each(gpu):
    """Four threads: systems of one workgroup and of several, both precisions."""
    ctxs = [_context(20, 21), _context(70, 61), _context(25, 22), _context(120, 90)]
    kinds = [(1, bief.PREC_FP64), (1, bief.PREC_MIXED), (7, bief.PREC_MIXED)]
    want = [[solve(*k)[0] for k in kinds] for _, solve in ctxs]
    bad = []

    def run(i):
        for _ in range(25):
            for k, w in zip(kinds, want[i]):
                x, on = ctxs[i][1](*k)
                if on is not True or not np.array_equal(x, w):
                    bad.append((i, k))

    ts = [threading.Thread(target=run, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad, bad
    for ctx, _ in ctxs:
        ctx.close()
