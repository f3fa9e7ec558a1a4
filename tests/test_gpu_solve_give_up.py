"""One handle solves different systems in turn while its one-kernel solve's waits
are bounded at times from 10 ns to 30 us, about as long as a hand-over takes, so
that solves give up at any of their hand-overs, the last one among them: there
every model may be finished and its solution stored while some blocks have left.
Whatever a solve leaves behind, it and the next one (which runs to its end) give
the kernel-per-step form's solution, bit for bit.  The systems differ in their
right-hand sides, so that a word left by one would be wrong for the next.
"""
import numpy as np
import pytest

from gpu_helpers import bits_equal, say
from adhv8_kraken_amd import mesh
from adhv8_kraken_amd.sw2 import SW2Model, default_opts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("cells", [(40, 20), (127, 63)])   # 4 and 32 blocks
def test_solves_after_a_give_up_at_any_hand_over(cells, precision):
    rng = np.random.default_rng(5)
    g = SW2Model(mesh.bumpy_channel(*cells), default_opts(precision=precision))
    g.shift(); g.init(); g.resid()
    diag, offd, rhs = g.load()
    systems = [rhs * (1.0 + 0.5 * rng.standard_normal(rhs.size)) for _ in range(4)]

    def solve(k, wait):
        g.set_solve_wait(wait)
        g.set_system(diag, offd, systems[k])
        g.linear_sys_setup()
        return g.linear_sys_solve()

    want = [solve(k, -1) for k in range(4)]
    say(f"  {cells} precision {precision}: {[w[2] for w in want]} iterations")
    for n, wait in enumerate(np.exp(rng.uniform(0.0, np.log(3000.0), 300)).astype(int)):
        for k, w in ((n % 4, int(wait)), ((n + 1) % 4, 1000000)):
            v, x, it = solve(k, w)
            assert (v, it) == (want[k][0], want[k][2]), f"solve {n}, wait {w}"
            assert bits_equal(x, want[k][1]), f"solve {n}, wait {w}"
    g.close()
