"""The wet / general triangle lists and the fused residual norms at the edges of
their block counts: one triangle block and its remainder, 1,024 count blocks (a
block's first round of counts to add up) and more, and 65,536 triangles, up to
which both lists share a launch.  On a partly dry floodplain,
where both lists are filled, residual and opening norms equal the oracle's (the
residual bit for bit, the l2 norm to the rounding of another summation order:
N eps of its square).
"""
import numpy as np
import pytest

from gpu_helpers import bits_equal, pair, say
from adhv8_kraken_amd import mesh
from adhv8_kraken_amd.sw2 import default_opts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(1, 1), (16, 8), (13, 10), (256, 128), (256, 129), (512, 256), (640, 250)])
def test_lists_and_norms_equal_oracle(cells):
    p = mesh.floodplain(*cells)
    o, g = pair(p, None, default_opts(max_nonlin_it=1, tol_nonlin=1e30))
    o.shift(); o.init()
    g.shift(); g.init()
    r = o.resid()
    say(f"  {p.nelems2d} triangles")
    assert bits_equal(r, g.resid())
    head, old = (np.asarray(a) for a in (o.get_state()[0], o.get_state()[2]))
    rep = g.newton()
    live = np.repeat(np.minimum(head, old) > 0.0, 3)
    l2 = np.sqrt(np.sum(r.astype(np.longdouble) ** 2) / r.size)
    assert rep["hist_max"][0] == (np.abs(r[live]).max() if live.any() else 0.0)
    assert abs(rep["hist_l2"][0] - l2) <= r.size * 2.3e-16 * l2
