"""The tiled band LU's sweeps with more bands than the GPU holds workgroups: 900
models factored from both ends, 1,800 bands, where the bands from the start
wait for those from the end.  Every model takes the step it takes alone, bit for
bit.
"""
import pytest

from gpu_helpers import bits_equal, say
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
