"""The tiled band LU's sweeps with so many bands that each has one workgroup, which
takes its rows in order without tickets: against an exact LU, and against the
models alone (several workgroups a band) bit for bit.
"""
import numpy as np
import pytest

from gpu_helpers import bits_equal, say
from test_gpu_lu_tiles import _system
from adhv8_kraken_amd import mesh
from adhv8_kraken_amd.sw2 import SW2Ensemble, SW2Model, default_opts

pytestmark = pytest.mark.gpu


# blocks of 63 DOFs, all one tile; the same with a last one of two; 72 DOFs; 498 DOFs in eight
# tiles, three from each end; 609 DOFs in bands wider than half of them
@pytest.mark.parametrize("ncx,ncy,nblock", [(300, 20, 301), (300, 20, 300), (300, 20, 260), (2400, 8, 130),
                                            (259, 200, 257)])
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


def test_reaches_longer_than_the_hand_over_ring():
    """132 models of 4,326 DOFs, 2,166 wide: 264 bands, rows of up to 34 tiles."""
    kinds = [mesh.bumpy_channel(1, 720, seed=k) for k in range(3)]
    opts = default_opts(preconditioner=1, nblock=1, lu_tiled=1, max_nonlin_it=3, tol_nonlin=1e-9)
    e = SW2Ensemble([kinds[k % 3] for k in range(132)], opts)
    rs = e.timestep()
    for k, p in enumerate(kinds):
        g = SW2Model(p, opts)
        r, s = g.timestep(), g.get_state()[:2]
        say(f"  model {k}: {r['iterations']} iterations")
        for i in range(k, 132, 3):
            assert r["iterations"] == rs[i]["iterations"] and bits_equal(r["hist_max"], rs[i]["hist_max"])
            assert all(bits_equal(a, b) for a, b in zip(s, e.get_state(i)))
        g.close()
    e.close()
