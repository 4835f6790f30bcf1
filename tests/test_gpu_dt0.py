"""gam_set_dt0 on a context that has already run: CalcDT's cap of 10 dt0
(step.F90:164-166) and its limDT0 check take the new value in every route a
step has -- single, replayed from a graph, of an ensemble -- and an adjoint
that puts recorded clocks back leaves it alone.

The cap is a product of two doubles, the same on both sides: equal.
"""
import numpy as np
import pytest

from helpers import box_case, shell_case
from mage_amd import gamhip

pytestmark = pytest.mark.gpu


def _make(kind):
    g = shell_case((16, 11, 13), state="mhd")[0] if kind == "shell" else box_case((16, 9, 11))[0]
    g.init_run()
    g.run(4)
    return g, g.get_time()[1] / 40


@pytest.mark.parametrize("kind", ["box", "shell"])
@pytest.mark.parametrize("route", ["run", "step", "advance", "ensemble"])
def test_new_dt0_binds(kind, route):
    g, dt0 = _make(kind)
    e = gamhip.GamEnsemble([g]) if route == "ensemble" else None
    if e:
        e.run(2)
    assert g.get_time()[1] > 10 * dt0
    for q in (1.0, 0.5):            # and once more, after graphs of the first
        g.set_dt0(q * dt0)
        assert g.get_dt0() == q * dt0
        if e:
            e.run(2)
        elif route == "run":
            g.run(2)
        elif route == "step":
            g.step()
        else:
            g.advance_model(0.0)
        assert g.get_time()[1] == 10.0 * (q * dt0)
    g.set_dt0(0.0)                  # no reference step: no cap
    if e:
        e.run(2)
        e.close()
    else:
        g.run(2)
    assert g.get_time()[1] > 10 * dt0
    g.close()


def test_new_dt0_fails_the_check_in_a_replayed_pair():
    g, dt0 = _make("box")
    g.set_dt0(1e6 * dt0)            # dt / dt0 = 4e-5 <= limDT0 = 1e-3
    with pytest.raises(gamhip.GamError) as ei:
        g.run(2)
    assert ei.value.code == -4    # GAM_E_DT_BAD
    g.close()


def test_adjoint_leaves_dt0_alone():
    g, dt0 = _make("shell")
    w = np.ones(g.cshape, order="F")
    adj = gamhip.GamAdjoint(g, 4, 2)
    adj.set_weights(w)
    adj.forward()
    g.set_dt0(dt0)
    adj.backward()
    adj.close()
    g.step()
    assert g.get_time()[1] == 10.0 * dt0
    g.close()
