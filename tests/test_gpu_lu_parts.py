"""The tiled band LU where a step's window tiles are more than the GPU takes at once:
the panels are formed by a launch of their own and the window takes them from memory.
Against an exact LU, against the models alone (few tiles: one launch a panel) bit
for bit, and its rate.
"""
import time

import numpy as np
import pytest

from gpu_helpers import bits_equal, say
from test_gpu_lu_tiles import _system
from adhv8_kraken_amd import mesh
from adhv8_kraken_amd.sw2 import SW2Ensemble, SW2Model, default_opts

pytestmark = pytest.mark.gpu


# windows of 5 tiles a side with the last one part full and of up to 3; blocks from both ends
# (879 DOFs) and from one (576; 165, all of it the first panel's window; the last one 381)
@pytest.mark.parametrize("ncx,ncy,nblock", [(60, 100, 21), (60, 100, 32), (80, 61, 90)])
def test_apply_is_the_block_inverse(ncx, ncy, nblock):
    """The system is diagonally dominant (condition below 10), so M^-1 v is the exact
    block inverse's to 1e-13 of its largest entry, as in test_gpu_lu_tiles.py."""
    import scipy.sparse as sp
    import scipy.sparse.linalg as sl
    p = mesh.bumpy_channel(ncx, ncy, seed=7)
    N = p.nnodes
    g = SW2Model(p, default_opts(preconditioner=1, nblock=nblock, lu_tiled=1))
    diag, offd, A = _system(g, 3)
    v = np.random.default_rng(5).uniform(-1.0, 1.0, 3 * N)
    g.set_system(diag, offd, v)
    s = g.linear_sys_setup()
    S = (sp.diags(s) @ A @ sp.diags(s)).tocoo()
    block = lambda i: np.minimum(i // 3 // (N // nblock), nblock - 1)   # noqa: E731
    keep = block(S.row) == block(S.col)
    inside = sp.csc_matrix((S.data[keep], (S.row[keep], S.col[keep])), shape=S.shape)
    ref = sl.splu(inside, permc_spec="NATURAL").solve(v)
    for rep in range(2):
        err = np.abs(g.precond_apply(v) - ref).max() / np.abs(ref).max()
        say(f"  {ncx}x{ncy} cells in {nblock} blocks, apply {rep}: {err:.1e}")
        assert err < 1e-13
    g.close()


def test_an_ensemble_takes_the_steps_of_its_models_alone():
    """Bands of no window, of one tile a side and of two to seven, from one end and
    from both, over 768 tiles in all until models have converged and fewer after."""
    cells = [(3, 1), (64, 1), (75, 1), (200, 4), (30, 40), (12, 130)]
    kinds = [mesh.bumpy_channel(*c, seed=k) for k, c in enumerate(cells)]
    ps = [kinds[k % 6] for k in range(48)]
    opts = default_opts(preconditioner=1, nblock=1, lu_tiled=1, max_nonlin_it=12, tol_nonlin=1e-9)
    e = SW2Ensemble(ps, opts)
    rs = e.timestep()
    for k, p in enumerate(kinds):
        g = SW2Model(p, opts)
        r, s = g.timestep(), g.get_state()[:2]
        say(f"  {3 * p.nnodes} DOFs: {r['iterations']} iterations")
        for i in range(k, 48, 6):
            assert r["iterations"] == rs[i]["iterations"] and bits_equal(r["hist_max"], rs[i]["hist_max"])
            assert all(bits_equal(a, b) for a, b in zip(s, e.get_state(i)))
        g.close()
    e.close()


def test_rate_with_many_wide_bands():
    """1000 x 500 cells in 16 blocks, 1,506 DOFs wide.  The factorisation's 2 m w^2
    operations took 360 ms (19 TFLOP/s) in parts and 623 (11) where every tile forms
    its own panels; four iterations, nine applications, 136 ms with a sweep
    workgroup a CU and 185 with two: the lines lie halfway."""
    p = mesh.bumpy_channel(1000, 500)
    g = SW2Model(p, default_opts(preconditioner=1, nblock=16, max_lin_it=4, lin_rtol=0.0, lin_atol=0.0))
    ops, setup, solve = 2.0 * 3 * p.nnodes * 1506.0 ** 2, [], []
    for _ in range(3):
        g.shift()
        g.init()
        g.resid()
        g.load()
        t0 = time.perf_counter()
        g.linear_sys_setup()
        t1 = time.perf_counter()
        g.linear_sys_solve()
        setup.append(t1 - t0)
        solve.append(time.perf_counter() - t1)
    say(f"  set-up {1e3 * min(setup):.0f} ms, {ops / min(setup) / 1e12:.1f} TFLOP/s; solve {1e3 * min(solve):.0f} ms")
    g.close()
    assert ops / min(setup) > 14.5e12
    assert min(solve) < 0.158
