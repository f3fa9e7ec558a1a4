"""The one-kernel block-Jacobi BiCGSTAB against the kernel-per-step form: the
same operations in the same order, so solution, iteration count and time step
agree bit for bit.  At one block and its edges, at the sizes where the number of
blocks a CU changes (256 blocks in FP64) and where the form ends (512), with
three to eight neighbours a node, and when the kernel's waits give up.
"""
import numpy as np
import pytest

from gpu_helpers import bits_equal, say
from adhv8_kraken_amd import mesh
from adhv8_kraken_amd.sw2 import SW2Ensemble, SW2Model, default_opts

pytestmark = pytest.mark.gpu
PER_STEP, NO_WAIT, DEFAULT = -1, 0, 30000


def _flipped(p, every):
    """The mesh with the diagonals of some quads turned: nodes of degree 7 and 8."""
    e = p.e2d.reshape(-1, 3).copy()
    for k in every(len(e) // 2):
        (a, b, c), d = e[2 * k], e[2 * k + 1][2]
        e[2 * k], e[2 * k + 1] = (a, b, d), (b, c, d)
    p.e2d = e.reshape(p.e2d.shape).astype(p.e2d.dtype)
    return p


CASES = {
    "1x1": lambda: mesh.bumpy_channel(1, 1),                                      # 3 neighbours
    "40x1": lambda: mesh.bumpy_channel(40, 1),                                    # 4 neighbours
    "15x15": lambda: mesh.bumpy_channel(15, 15),                                  # 256 nodes, one block
    "16x15": lambda: mesh.bumpy_channel(16, 15),                                  # 16 nodes in the second block
    "63x31-degree7": lambda: _flipped(mesh.bumpy_channel(63, 31), lambda n: [n // 2 + 15]),
    "64x32-degree8": lambda: _flipped(mesh.bumpy_channel(64, 32), lambda n: [k for k in range(n) if (k // 64 + k) % 2]),
    "255x255": lambda: mesh.bumpy_channel(255, 255),                              # 256 blocks
    "256x255": lambda: mesh.bumpy_channel(256, 255),                              # 257 blocks
    "511x255": lambda: mesh.bumpy_channel(511, 255),                              # 512 blocks
    "512x255": lambda: mesh.bumpy_channel(512, 255),                              # 513: the other form
}


def _solve(p, precision, wait, guess):
    g = SW2Model(p, default_opts(precision=precision))
    g.set_solve_wait(wait)
    g.shift(); g.init(); g.resid(); g.load()
    g.linear_sys_setup(guess)
    first = g.linear_sys_solve()
    g.set_opts(default_opts(precision=precision, max_nonlin_it=3, tol_nonlin=1e-9))
    r = g.timestep()
    state = g.get_state()
    g.close()
    return first, r["iterations"], r["lin_its"], r["hist_max"], state


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("name", sorted(CASES))
def test_one_kernel_solve_equals_kernel_per_step(name, precision):
    p = CASES[name]()
    guess = np.random.default_rng(3).normal(0.0, 1e-3, 3 * p.nnodes)
    (v0, x0, it0), n0, lin0, h0, s0 = _solve(p, precision, PER_STEP, guess)
    say(f"  {name} precision {precision}: {p.nnodes} nodes, {it0} iterations")
    assert it0 > 0 and np.isfinite(x0).all()
    for wait in (DEFAULT, NO_WAIT):
        (v, x, it), n, lin, h, s = _solve(p, precision, wait, guess)
        assert (v, it, n, lin) == (v0, it0, n0, lin0)
        assert bits_equal(x, x0) and bits_equal(h, h0)
        assert all(bits_equal(a, b) for a, b in zip(s, s0))


@pytest.mark.parametrize("precision", [0, 1])
def test_one_kernel_solve_of_more_models_than_fit_at_once(precision):
    ps = [mesh.bumpy_channel(20 + 7 * (k % 9), 30 + 11 * (k % 5), seed=k) for k in range(60)]
    runs = []
    for wait in (PER_STEP, DEFAULT, NO_WAIT):
        g = SW2Ensemble(ps, default_opts(precision=precision, max_nonlin_it=6, tol_nonlin=1e-7))
        g.set_solve_wait(wait)
        r = g.timestep()
        runs.append((r, [g.get_state(k) for k in range(len(ps))]))
        g.close()
    say(f"  60 models, {sum((p.nnodes + 255) // 256 for p in ps)} blocks")
    for r, s in runs[1:]:
        assert [q["lin_its"] for q in r] == [q["lin_its"] for q in runs[0][0]]
        for a, b in zip(s, runs[0][1]):
            assert all(bits_equal(x, y) for x, y in zip(a, b))


def test_models_of_three_threads_that_do_not_fit_together():
    """Three handles stepped by three threads at once, 315 blocks each of the 512
    that the GPU holds: whichever solves find the CUs taken give up and are
    repeated, and every model ends where it ends alone, bit for bit."""
    import threading
    ps = [mesh.bumpy_channel(401, 199, seed=k) for k in range(3)]
    opts = default_opts(max_nonlin_it=3, tol_nonlin=1e-9)

    def steps(p):
        g = SW2Model(p, opts)
        for _ in range(3):
            g.timestep()
        s = g.get_state()
        g.close()
        return s

    alone = [steps(p) for p in ps]
    together = [None] * 3

    def run(k):
        together[k] = steps(ps[k])

    threads = [threading.Thread(target=run, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(alone, together):
        assert b is not None and all(bits_equal(x, y) for x, y in zip(a, b))
