"""The wet / general triangle lists where their count blocks are first added up by
runs: 6,144 count blocks (1,572,864 triangles), the last mesh without, and one
row of cells more, with a last run and a last block that are not full.  Residual
and lists as in test_gpu_split_lists.py: on a partly dry floodplain the residual
equals the oracle's bit for bit, which takes every triangle in exactly one list.
"""
import pytest

from gpu_helpers import bits_equal, pair, say
from adhv8_kraken_amd import mesh
from adhv8_kraken_amd.sw2 import default_opts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(1024, 768), (1025, 768)])
def test_residual_equals_oracle_on_both_sides_of_the_runs(cells):
    p = mesh.floodplain(*cells)
    o, g = pair(p, None, default_opts())
    o.shift(); o.init()
    g.shift(); g.init()
    r = o.resid()
    say(f"  {p.nelems2d} triangles, {(p.nelems2d + 255) // 256} count blocks")
    assert bits_equal(r, g.resid())
    g.close()
