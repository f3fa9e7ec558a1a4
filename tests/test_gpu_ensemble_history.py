"""The whole residual history of an ensemble's models over three steps, the norm
of the correction among it, against each model's own run, bit for bit.  The
models finish at different iterations, so the others' set-ups and solves must
leave a finished model's correction alone: its norm opens the next step's
history.  With the one-kernel solve and with a kernel per step, in every form.
"""
import pytest

from gpu_helpers import bits_equal, say
from adhv8_kraken_amd import mesh
from adhv8_kraken_amd.sw2 import SW2Ensemble, SW2Model, default_opts

pytestmark = pytest.mark.gpu

FORMS = {"fp64": dict(precision=0), "refined": dict(precision=1), "fp32": dict(precision=2),
         "direct": dict(precision=0, preconditioner=1, nblock=1, lu_tiled=1),
         "blocks": dict(precision=0, preconditioner=1, nblock=4, lu_tiled=1)}


@pytest.mark.parametrize("wait", [30000, -1])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_history_of_models_that_finish_apart(form, wait):
    ps = [mesh.bumpy_channel(*c, seed=k) for k, c in enumerate([(40, 20), (30, 12), (60, 30), (17, 23)])]
    tols = [1e-2, 1e-7, 1e-4, 1e-6]
    e = SW2Ensemble(ps, default_opts(max_nonlin_it=12, **FORMS[form]))
    e.set_solve_wait(wait)
    for i, t in enumerate(tols):
        e.set_tol(i, t)
    together = [e.timestep() for _ in range(3)]
    its = [[r["iterations"] for r in rs] for rs in together]
    say(f"  {form}: iterations {its}")
    assert any(len(set(k)) > 1 for k in its), "the models finish together: nothing is tested"
    for i, (p, t) in enumerate(zip(ps, tols)):
        g = SW2Model(p, default_opts(max_nonlin_it=12, tol_nonlin=t, **FORMS[form]))
        g.set_solve_wait(wait)
        for s in range(3):
            a, b = g.timestep(), together[s][i]
            for key in ("hist_max", "hist_l2", "hist_inc", "hist_lin_it"):
                assert bits_equal(a[key], b[key]), f"model {i}, step {s}, {key}: {a[key]} {b[key]}"
        g.close()
    e.close()
