"""The autotuner where the lists and the edges share a launch (up to 32,768
triangles for the Jacobian, 65,536 for the residual) and just above: the shapes it
keeps make a load and a residual, launches of all their parts, no slower than the
defaults' (within a tenth and 2 us of host timing), on wet and on half dry meshes, and change no bit of
the system.
"""
import ctypes as C
import time

import pytest

from gpu_helpers import bits_equal, say
from adhv8_kraken_amd import mesh
from adhv8_kraken_amd.sw2 import SW2Model, default_opts

pytestmark = pytest.mark.gpu
NULL = C.POINTER(C.c_double)()


def _us(call, n=80):
    ts = []
    for _ in range(n):
        t0 = time.perf_counter()
        assert call() == 0
        ts.append(time.perf_counter() - t0)
    ts.sort()
    return 1e6 * ts[n // 8]


@pytest.mark.parametrize("make", [mesh.bumpy_channel, mesh.floodplain])
@pytest.mark.parametrize("cells", [(40, 20), (121, 57), (128, 128), (181, 181), (182, 181)])
def test_tuned_shapes_are_no_slower_in_the_launch_that_runs(make, cells):
    g = SW2Model(make(*cells), default_opts())
    g.shift(); g.init(); g.resid()
    load, resid = (lambda: g.L.adh_sw2_hip_load(g.h, NULL, NULL, NULL)), (lambda: g.L.adh_sw2_hip_resid(g.h, NULL))
    r0, s0 = g.resid(), g.load()
    before = _us(load), _us(resid)
    chosen = g.autotune(5)
    after = _us(load), _us(resid)
    say(f"  {make.__name__} {cells}: load {before[0]:.1f} -> {after[0]:.1f} us, residual {before[1]:.1f} -> "
        f"{after[1]:.1f}; {chosen}")
    assert after[0] < 1.1 * before[0] + 2.0
    assert after[1] < 1.1 * before[1] + 2.0
    assert bits_equal(r0, g.resid())
    assert all(bits_equal(a, b) for a, b in zip(s0, g.load()))
    g.close()
