"""The tiled band LU's sweeps with more bands than the GPU holds workgroups: 900
models factored from both ends, 1,800 bands, where the bands from the start
wait for those from the end.  Every model takes the step it takes alone, bit for
bit.  And with more bands than a grid has rows.
"""
import numpy as np
import pytest

from gpu_helpers import bits_equal, say
from test_gpu_lu_tiles import _system
from adhv8_kraken_amd import mesh
from adhv8_kraken_amd.sw2 import SW2Ensemble, SW2Model, default_opts

pytestmark = pytest.mark.gpu


def test_more_two_ended_bands_than_workgroups_fit():
    kinds = [mesh.bumpy_channel(*c, seed=k) for k, c in enumerate([(65, 1), (75, 1), (64, 1)])]   # two, two, one band
    ps = [kinds[k % 2 if k % 50 else 2] for k in range(900)]
    opts = default_opts(preconditioner=1, nblock=1, max_nonlin_it=3, tol_nonlin=1e-9)
    e = SW2Ensemble(ps, opts)
    rs = e.timestep()
    for kind in kinds:
        g = SW2Model(kind, opts)
        r, s = g.timestep(), g.get_state()[:2]
        at = [i for i, p in enumerate(ps) if p is kind]
        say(f"  {3 * kind.nnodes} DOFs: {r['iterations']} iterations, {len(at)} models")
        for i in at:
            assert rs[i]["iterations"] == r["iterations"] and bits_equal(rs[i]["hist_max"], r["hist_max"])
        for i in at[::40] + at[-1:]:
            assert all(bits_equal(a, b) for a, b in zip(s, e.get_state(i)))
        g.close()
    e.close()


@pytest.mark.parametrize("blocks", [32769, 66000])
def test_more_bands_than_a_grid_has_rows(blocks):
    """Blocks of a few nodes, one more than a launch takes (the last block holds the
    1,392 nodes that are left over, factored from both ends) and more than HIP's
    grids have rows.  The system is diagonally dominant (condition below 10), so
    M^-1 v is the exact block inverse's to 1e-13 of its largest entry, as in
    test_gpu_lu_tiles.py."""
    import scipy.sparse as sp
    import scipy.sparse.linalg as sl
    p = mesh.bumpy_channel(659, 299)   # 198,000 nodes
    N = p.nnodes
    g = SW2Model(p, default_opts(preconditioner=1, nblock=blocks, lu_tiled=1))
    diag, offd, A = _system(g, 3)
    v = np.random.default_rng(5).uniform(-1.0, 1.0, 3 * N)
    g.set_system(diag, offd, v)
    s = g.linear_sys_setup()
    S = (sp.diags(s) @ A @ sp.diags(s)).tocoo()
    block = lambda i: np.minimum(i // 3 // (N // blocks), blocks - 1)   # noqa: E731
    keep = block(S.row) == block(S.col)
    inside = sp.csc_matrix((S.data[keep], (S.row[keep], S.col[keep])), shape=S.shape)
    ref = sl.splu(inside, permc_spec="NATURAL").solve(v)
    for rep in range(2):
        err = np.abs(g.precond_apply(v) - ref).max() / np.abs(ref).max()
        say(f"  {blocks} blocks, apply {rep}: {err:.1e}")
        assert err < 1e-13
    g.close()
