"""The tiled band LU at the edges of its tiles: one tile, blocks that end on a
tile and one DOF past it, bands narrower than a tile, reaches longer than the
sweep's hand-over ring, several node blocks, and a pivot that takes the guard.

The system is random and diagonally dominant on a mesh's pattern, so its LU
needs no pivoting and its condition number is below 10: M^-1 v of two exact
factorisations in FP64 differs by a small multiple of cond * eps * (DOFs a row
couples to, <= 21), bounded here by 1e-13 of the largest entry.
"""
import numpy as np
import pytest

from gpu_helpers import bits_equal, say
from adhv8_kraken_amd import mesh
from adhv8_kraken_amd.sw2 import SW2Ensemble, SW2Model, default_opts

pytestmark = pytest.mark.gpu


def _system(g, seed):
    """Random diagonally dominant blocks on the model's pattern, and the CSR of it."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    N = g.N
    rp, col = g.pattern()
    row = np.repeat(np.arange(N), np.diff(rp))
    offd = rng.uniform(-1.0, 1.0, 9 * len(col)) / 21.0
    diag = rng.uniform(-1.0, 1.0, 9 * N) / 21.0
    for v in range(3):
        diag[4 * v::9] = rng.uniform(2.0, 4.0, N) * rng.choice([-1.0, 1.0], N)
    i, j = np.tile(np.repeat(np.arange(3), 3), N), np.tile(np.arange(3), 3 * N)
    io, jo = np.tile(np.repeat(np.arange(3), 3), len(col)), np.tile(np.arange(3), 3 * len(col))
    A = sp.csr_matrix((np.concatenate([diag, offd]),
                       (np.concatenate([np.repeat(3 * np.arange(N), 9) + i, np.repeat(3 * row, 9) + io]),
                        np.concatenate([np.repeat(3 * np.arange(N), 9) + j, np.repeat(3 * col, 9) + jo]))),
                      shape=(3 * N, 3 * N))
    return diag, offd, A


# (cells along, cells across, node blocks): DOFs 12 (part of one tile), 192 = 3 tiles in a
# band of 17, 195, 693, reaches of 33 and 34 tiles, blocks of 64 and 128 DOFs and their remainders;
# 390, 396 and 456 DOFs: the last block in one band, three panels from each end with one shared panel and with two
@pytest.mark.parametrize("ncx,ncy,nblock", [(1, 1, 1), (15, 3, 1), (12, 4, 1), (20, 10, 1), (4, 700, 1), (3, 720, 1),
                                            (20, 10, 2), (42, 5, 5), (31, 20, 9),
                                            (64, 1, 1), (65, 1, 1), (75, 1, 1)])
def test_apply_is_the_block_inverse(ncx, ncy, nblock):
    import scipy.sparse as sp
    import scipy.sparse.linalg as sl
    p = mesh.bumpy_channel(ncx, ncy, seed=7)
    g = SW2Model(p, default_opts(preconditioner=1, nblock=nblock, lu_tiled=1))
    diag, offd, A = _system(g, 3)
    say(f"tiled LU {ncx}x{ncy} cells, {3 * p.nnodes} DOFs in {nblock} blocks")
    v = np.random.default_rng(5).uniform(-1.0, 1.0, 3 * p.nnodes)
    g.set_system(diag, offd, v)
    s = g.linear_sys_setup()
    S = sp.diags(s) @ A @ sp.diags(s)
    inc, N = p.nnodes // nblock, p.nnodes
    for rep in range(2):   # twice: the sweeps' tickets and ready values start afresh
        y = g.precond_apply(v)
        ref = np.empty(3 * N)
        for b in range(nblock):
            a, e = 3 * b * inc, 3 * N if b == nblock - 1 else 3 * (b + 1) * inc
            ref[a:e] = sl.splu(S[a:e, a:e].tocsc()).solve(v[a:e])
        err = np.abs(y - ref).max() / np.abs(ref).max()
        say(f"  apply {rep}: {err:.2e}")
        assert err < 1e-13
    g.close()


@pytest.mark.parametrize("node", [0, 21, 100, 230])
def test_backward_sweep_divides_by_the_pivot_itself(node):
    """A node whose row is too small for the scaling keeps a scaled pivot of
    1e-17, below the guard: nothing couples to it, so the elimination is that
    of the rest and its solution is v / pivot, not v / SMALL."""
    import scipy.sparse as sp
    import scipy.sparse.linalg as sl
    p = mesh.bumpy_channel(20, 10, seed=7)
    g = SW2Model(p, default_opts(preconditioner=1, nblock=1, lu_tiled=1))
    diag, offd, A = _system(g, 3)
    rp, col = g.pattern()
    row = np.repeat(np.arange(g.N), np.diff(rp))
    offd = offd.reshape(-1, 9)
    offd[(row == node) | (col == node)] = 0.0
    tiny = 1e-17 * 2.220446049250313e-16
    diag.reshape(-1, 9)[node] = np.eye(3).ravel() * tiny
    v = np.random.default_rng(5).uniform(0.5, 1.0, 3 * p.nnodes)
    g.set_system(diag, offd.ravel(), v)
    s = g.linear_sys_setup()
    y = g.precond_apply(v)
    mine = np.arange(3 * node, 3 * node + 3)
    say(f"guarded node {node}: scaled pivots {tiny * s[mine] ** 2}, y {y[mine]}")
    assert np.all(np.abs(y[mine] * (tiny * s[mine] ** 2) / v[mine] - 1.0) < 1e-14)
    rest = np.setdiff1d(np.arange(3 * p.nnodes), mine)
    S = (sp.diags(s) @ A @ sp.diags(s)).tocsr()[rest][:, rest]
    ref = sl.splu(S.tocsc()).solve(v[rest])
    assert np.abs(y[rest] - ref).max() < 1e-13 * np.abs(ref).max()
    g.close()


def test_models_of_one_band_and_of_two_factor_together():
    """One to 60 tiles, factored from one end and from both, in one ensemble:
    the bands meet their shared rows at one launch, and each model takes the
    steps it takes alone, bit for bit."""
    ps = [mesh.bumpy_channel(*c, seed=k) for k, c in enumerate([(3, 1), (64, 1), (65, 1), (75, 1), (200, 4), (30, 40)])]
    opts = default_opts(preconditioner=1, nblock=1, lu_tiled=1, max_nonlin_it=4, tol_nonlin=1e-9)
    e = SW2Ensemble(ps, opts)
    rs = e.timestep()
    for k, p in enumerate(ps):
        g = SW2Model(p, opts)
        r = g.timestep()
        say(f"  {3 * p.nnodes} DOFs: {r['iterations']} iterations")
        assert r["iterations"] == rs[k]["iterations"] and bits_equal(r["hist_max"], rs[k]["hist_max"])
        assert all(bits_equal(a, b) for a, b in zip(g.get_state()[:2], e.get_state(k)))
        g.close()
    e.close()
