"""Model%dt = 0, which a context has until gam_init_run or gam_set_time and
which gam_set_time accepts: the EMF's vDiff cap CFL edge / dt is then no cap
(fields.F90:288-517 divides by it), forward and in the transpose.

AdvanceMHD with its own dt on such a clock against the oracle: 1e-12
relative L-infinity, as in test_gpu_step.py.  A step of dt = 0 maps every
state to itself, so the gradient is the objective's own, w dP/dU (0 for
oState and the face fluxes): 1e-12 of its largest entry, the rounding of the
conversions to primitives and back.
"""
import numpy as np
import pytest

from helpers import box_case, compare_state, shell_case
from mage_amd import gamhip

pytestmark = pytest.mark.gpu


def _case(kind, rmeth):
    return shell_case((16, 11, 13), rmeth, state="mhd") if kind == "shell" else box_case((16, 9, 11), rmeth)


@pytest.mark.parametrize("rmeth", ["8CENT", "7UP"])
@pytest.mark.parametrize("kind", ["box", "shell"])
@pytest.mark.parametrize("form", ["lds", "direct"])
def test_advance_without_a_model_dt_matches_oracle(kind, form, rmeth):
    g, o, grid, st, p = _case(kind, rmeth)
    if form == "direct":
        plan = g.get_plan()
        for d in "ijk":
            plan["emf_" + d] = 9
        g.set_plan(plan)
    dt = g.init_run()
    o.init_run()
    g.step()
    o.step()
    dt = g.get_time()[1]
    g.set_time(o.M.t, 0.0, 1)
    o.M.dt = 0.0
    for _ in range(2):
        g.advance_mhd(dt)
        o.advance(dt)
        e = compare_state(g, o)
        assert max(e.values()) <= 1e-12, e
    g.close()


@pytest.mark.parametrize("rmeth", ["8CENT", "7UP"])
@pytest.mark.parametrize("kind", ["box", "shell"])
def test_gradient_of_a_step_of_no_length(kind, rmeth):
    g, o, grid, st, p = _case(kind, rmeth)
    g.init_run()
    t, dt, ts = g.get_time()
    g.set_time(t, 0.0, ts)
    N = (g.Nip, g.Njp, g.Nkp)
    inner = tuple(slice(4, 4 + n) for n in N)
    w = np.zeros(g.cshape, order="F")
    w[inner] = grid["volume"][inner]
    adj = gamhip.GamAdjoint(g, 1, 1)
    adj.set_weights(w)
    adj.forward()
    assert adj.step_dt(1)[0] == 0.0
    gS, gO, gM, gMO = adj.backward(fluxes=True)
    U = g.get_state()["Gas"][inner]
    v = U[..., 1:4] / U[..., :1]
    gm = p["gamma"] - 1
    want = np.concatenate([gm * 0.5 * np.sum(v * v, axis=-1, keepdims=True), -gm * v,
                           np.full(U.shape[:3] + (1,), gm)], axis=-1) * w[inner][..., None]
    big = float(np.max(np.abs(want)))
    for x in (gS[inner] - want, gO[inner], gM[inner], gMO[inner]):
        err = float(np.max(np.abs(x)))
        assert err <= 1e-12 * big
    adj.close()
    g.close()
