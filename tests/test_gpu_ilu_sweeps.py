"""The ILU(0) apply's two forms, a launch per sweep and a launch per colour, at
the edges of their units and of the rule between them (200,000 rows).

Small meshes: against the CPU factors (1e-12, as tests/test_gpu_ilu.py).  Large
ones: a matrix that couples nodes 2k and 2k + 1 only, whose ILU(0) has no fill
and is exact, against 6 x 6 solves; random and diagonally dominant, so the two
differ by a small multiple of its condition number (below 10) times eps, bounded
by 1e-13.  Repeated applies start from the state the one before left.
"""
import numpy as np
import pytest

from gpu_helpers import bits_equal, say
from adhv8_kraken_amd import mesh
from adhv8_kraken_amd.sw2 import SW2Model, default_opts
from oracle.ilu0 import BlockILU0, colour_order
from test_gpu_ilu import _scaled_system, _stepped

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(1, 1), (15, 15), (16, 15), (70, 31)])
def test_apply_matches_the_cpu_factors_at_unit_edges(cells):
    g = _stepped(mesh.bumpy_channel(*cells), 3, 0)
    D, O, rp, col = _scaled_system(g)
    color, ncolor = g.ilu_colors()
    M = BlockILU0(D, O, colour_order(color)[1])
    v = np.random.default_rng(1).uniform(-1, 1, 3 * g.N)
    y = [g.precond_apply(v) for _ in range(3)]
    ref = M.apply(v)
    say(f"  {g.N} nodes, {ncolor} colours: {np.abs(y[0] - ref).max() / np.abs(ref).max():.2e}")
    assert np.abs(y[0] - ref).max() <= 1e-12 * np.abs(ref).max()
    assert bits_equal(y[0], y[1]) and bits_equal(y[0], y[2])
    g.close()


def _wheel():
    """A 20 x 20 channel with one node of twelve neighbours: the edges around it
    turned towards it.  Its slice's rows hold more blocks than the LDS."""
    p = mesh.bumpy_channel(20, 20)
    e = [list(t) for t in p.e2d.reshape(-1, 3)]
    hub = p.nnodes // 2
    for t in [t for t in e if hub in t]:
        k = t.index(hub)
        a, b = t[(k + 1) % 3], t[(k + 2) % 3]
        u = next(x for x in e if x is not t and a in x and b in x)
        c = next(n for n in u if n not in (a, b))
        t[:] = [hub, a, c]
        u[:] = [hub, c, b]
    p.e2d = np.array(e, dtype=p.e2d.dtype).reshape(p.e2d.shape)
    return p


def test_factors_of_rows_beyond_the_lds():
    g = _stepped(_wheel(), 3, 0)
    D, O, rp, col = _scaled_system(g)
    assert np.diff(rp).max() == 12
    M = BlockILU0(D, O, colour_order(g.ilu_colors()[0])[1])
    v = np.random.default_rng(1).uniform(-1, 1, 3 * g.N)
    ref = M.apply(v)
    assert np.abs(g.precond_apply(v) - ref).max() <= 1e-12 * np.abs(ref).max()
    g.close()


@pytest.mark.parametrize("cells", [(440, 440), (455, 450)])
def test_apply_is_exact_without_fill_on_both_sides_of_the_rule(cells):
    g = SW2Model(mesh.bumpy_channel(*cells), default_opts(preconditioner=3))
    N = g.N
    rp, col = g.pattern()
    row = np.repeat(np.arange(N), np.diff(rp))
    rng = np.random.default_rng(2)
    diag = rng.uniform(-1.0, 1.0, (N, 9)) / 21.0
    diag[:, [0, 4, 8]] = rng.uniform(2.0, 4.0, (N, 3))
    offd = np.where((row // 2 == col // 2)[:, None], rng.uniform(-1.0, 1.0, (len(col), 9)) / 3.0, 0.0)
    v = rng.uniform(-1.0, 1.0, 3 * N)
    g.set_system(diag.ravel(), offd.ravel(), v)
    s = g.linear_sys_setup()
    y = [g.precond_apply(v) for _ in range(2)]
    A = np.zeros((N // 2, 6, 6))
    for h in range(2):
        A[:, 3 * h:3 * h + 3, 3 * h:3 * h + 3] = diag[h:2 * (N // 2):2].reshape(-1, 3, 3)
        pair = (row // 2 == col // 2) & (row % 2 == h)
        A[row[pair] // 2, 3 * h:3 * h + 3, 3 - 3 * h:6 - 3 * h] = offd[pair].reshape(-1, 3, 3)
    s6 = s[:6 * (N // 2)].reshape(-1, 6)
    ref = np.linalg.solve(A * s6[:, :, None] * s6[:, None, :], v[:6 * (N // 2)].reshape(-1, 6, 1)).ravel()
    err = np.abs(y[0][:len(ref)] - ref).max() / np.abs(ref).max()
    say(f"  {N} nodes: {err:.2e}")
    assert err <= 1e-13
    assert bits_equal(y[0], y[1])
    g.close()
