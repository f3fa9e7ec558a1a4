"""Which form an ensemble's solve takes: models of just over half of the GPU's places
would run one at a time in the one-kernel form and go to the kernel-per-step
form; FP64 models of just over half of the places at one block a CU run at two.
On both sides of each line the states are the kernel-per-step form's, bit for
bit, and a step takes at most 1.05 times that form's time (24 models of 260
blocks took 1.09 times as long in one kernel).
"""
import time

import pytest

from gpu_helpers import bits_equal, say
from adhv8_kraken_amd import mesh
from adhv8_kraken_amd.sw2 import YES, SW2Ensemble, default_opts

pytestmark = pytest.mark.gpu


# models, cells: blocks of 256 nodes a model 128, 130, 256, 260, 450
@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("n,cells", [(8, (285, 113)), (24, (286, 115)), (6, (404, 161)), (24, (407, 162)), (6, (535, 214))])
def test_form_by_how_the_models_fill_the_gpu(n, cells, precision):
    ps = [mesh.bumpy_channel(*cells, seed=k) for k in range(n)]
    e = SW2Ensemble(ps, default_opts(precision=precision, max_nonlin_it=1, tol_nonlin=1e30))

    def step(wait):
        for i, p in enumerate(ps):
            e.set_state(i, p.head0, p.vel0, p.head0, p.vel0, p.head0, p.vel0)
        e.set_solve_wait(wait)
        e.get_state(0)
        t0 = time.perf_counter()
        rs = e.timestep()
        t = time.perf_counter() - t0
        assert all(r["verdict"] == YES for r in rs)
        return t

    step(-1)
    want = [e.get_state(i) for i in range(n)]
    both = [(step(-1), step(30000)) for _ in range(8)]   # by turns; the last one is the default form's
    per_step, t = (min(k) for k in zip(*both))
    say(f"  {n} models of {(ps[0].nnodes + 255) // 256} blocks, precision {precision}: {1e3 * t:.2f} ms, "
        f"a kernel per step {1e3 * per_step:.2f}")
    for i, w in enumerate(want):
        assert all(bits_equal(a, b) for a, b in zip(w, e.get_state(i)))
    assert t < 1.05 * per_step
    e.close()
