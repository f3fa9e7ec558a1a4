"""An ensemble of more blocks than the GPU holds at once: the models wait in turn for
the ones before them, longer than the bound of a wait inside the one-kernel solve
(0.3 ms), and that time does not count.  With the default bound such a solve takes
the time it takes with a bound of 10 s, where a give-up would repeat all of it
as a kernel per step; and it gives the kernel-per-step form's states, bit for bit.
"""
import time

import pytest

from gpu_helpers import bits_equal, say
from adhv8_kraken_amd import mesh
from adhv8_kraken_amd.sw2 import YES, SW2Ensemble, default_opts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_waiting_for_the_models_before_does_not_end_a_solve(precision):
    ps = [mesh.bumpy_channel(507, 201, seed=k) for k in range(4)]   # 401 blocks each, 512 at once
    # one Newton iteration a step, accepted; 30 and more iterations in its solve
    opts = default_opts(precision=precision, max_nonlin_it=1, tol_nonlin=1e30, max_lin_it=150, lin_rtol=1e-13, lin_atol=0.0)
    e = SW2Ensemble(ps, opts)

    def step(wait):
        for i, p in enumerate(ps):
            e.set_state(i, p.head0, p.vel0, p.head0, p.vel0, p.head0, p.vel0)
        e.set_solve_wait(wait)
        e.get_state(0)
        t0 = time.perf_counter()
        rs = e.timestep()
        t = time.perf_counter() - t0
        assert all(r["verdict"] == YES and r["lin_its"] >= 30 for r in rs)
        return t

    step(-1)
    want = [e.get_state(i) for i in range(len(ps))]
    long = min(step(1000000000) for _ in range(3))
    default = min(step(30000) for _ in range(3))
    say(f"  precision {precision}: {1e3 * long:.2f} ms with a bound of 10 s, {1e3 * default:.2f} with 0.3 ms")
    assert default < 1.3 * long
    assert not any(bits_equal(w[0], p.head0) for w, p in zip(want, ps))
    for i, w in enumerate(want):
        assert all(bits_equal(a, b) for a, b in zip(w, e.get_state(i)))
    e.close()
