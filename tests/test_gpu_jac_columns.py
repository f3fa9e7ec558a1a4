"""The element Jacobian's column split at the edges of its rule: one column a
wave up to 7,264 triangles, three up to 131,040, nine above; a last group of
fewer than 32 triangles, and one triangle group in all; both sides of 32,768,
up to which both lists and the edges share a launch.  Every split computes
the same columns from the same inputs, so the assembled system equals the
lane-per-column kernel's bit for bit.
"""
import numpy as np
import pytest

from gpu_helpers import bits_equal, say
from adhv8_kraken_amd import mesh
from adhv8_kraken_amd.sw2 import SW2Model, default_opts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("cells", [(4, 4), (17, 1), (56, 64), (227, 16), (56, 65), (128, 128), (128, 129),
                                   (252, 260), (256, 256)])
def test_column_split_equals_lane_kernel(cells, precision):
    p = mesh.floodplain(*cells)
    out = []
    for layout in (0, 3):
        g = SW2Model(p, default_opts(precision=precision))
        t = g.get_tuning()
        t.layout[0] = t.layout[1] = layout
        g.set_tuning(t)
        g.shift()
        g.init()
        g.resid()
        out.append(g.load())
        g.close()
    say(f"  {2 * cells[0] * cells[1]} triangles, precision {precision}")
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.abs(a).max() > 0.0
        assert bits_equal(a, b)
