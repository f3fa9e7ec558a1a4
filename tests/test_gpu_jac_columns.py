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


def test_autotuned_jacobian_is_no_slower_than_the_default():
    """The autotuner's times are those of its launches: the shape it keeps runs
    as fast as it says (twice that at most, a single timing of a launch of 0.2
    ms) and no slower than the default's (within a quarter)."""
    g = SW2Model(mesh.bumpy_channel(400, 200), default_opts(precision=1))
    g.shift(); g.init(); g.resid()
    before = g.time_kernel(1, 20)
    chosen = g.autotune(3)
    after = g.time_kernel(1, 20)
    say(f"  default {before:.4f} ms, tuned {after:.4f} ms, {chosen['jac_wet']}")
    assert 0.5 * after < chosen["jac_wet"]["ms"] < 2.0 * after
    assert after < 1.25 * before
    assert 0.0 < chosen["res_wet"]["ms"] < 0.8 * chosen["jac_wet"]["ms"]
    g.close()
