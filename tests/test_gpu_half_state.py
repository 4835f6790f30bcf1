"""Steps that form the half state inside the fluxes and EMFs (from the third
step of a state on) against steps through the predictor and the oracle: the
half state handed out (gam_get_state of GAM_HFSTATE) whatever the route and
whatever happens to State and oState before it is asked for, and states
changed between steps, which go back to the predictor.

Tolerances (relative L-infinity): 1e-12 after a few steps, as in
test_gpu_step.py; equal where the same kernel forms both sides.
"""
import numpy as np
import pytest

from helpers import box_case, compare_state, rel_linf, shell_case
from mage_amd import gamhip, problems as pb

pytestmark = pytest.mark.gpu

TOL = 1e-12
HF = gamhip.GAM_HFSTATE
KEYS = ("Gas", "magFlux", "Bxyz")


def _case(kind, **over):
    if kind == "shell":
        return shell_case((24, 11, 13), state="mhd", **over)
    if kind.startswith("hydro"):
        return box_case((16, 9, 11), "8CENT" if kind == "hydro8" else "7UP", doMHD=0, **over)
    return box_case((16, 9, 11), "8CENT" if kind == "box8" else "7UP", **over)


def _worst(a, b):
    return max(rel_linf(a[k], b[k]) for k in KEYS)


@pytest.mark.parametrize("kind", ["box7", "box8", "shell", "hydro7", "hydro8"])
@pytest.mark.parametrize("route,lfm", [("step", 1), ("run4", 1), ("run5", 1), ("run5", 0), ("advance", 1),
                                       ("ensemble", 1)])
def test_half_state_of_the_last_step(kind, route, lfm):
    g, o, grid, st, p = _case(kind, doLFMLim=lfm)
    dt = g.init_run()
    o.init_run()
    n = 4 if route == "run4" else 5
    if route == "step":
        for _ in range(n):
            g.step()
    elif route == "advance":
        n = g.advance_model(3.5 * dt)       # however many steps that takes
        assert n > 2
    elif route == "ensemble":
        e = gamhip.GamEnsemble([g])
        e.run(2)
        e.run(3)
        e.close()
    else:
        g.run(n)
    for _ in range(n):
        o.step()
    assert max(compare_state(g, o).values()) <= TOL
    assert _worst(g.get_state(HF), o.half_state()) <= TOL
    g.run(2)
    o.step()
    o.step()
    assert max(compare_state(g, o).values()) <= TOL
    assert _worst(g.get_state(HF), o.half_state()) <= TOL
    g.close()


@pytest.mark.parametrize("after", ["init", "put_old", "put_new", "bcs", "grid", "init_step", "tune"])
def test_half_state_outlives_its_states(after):
    a, _, grid, st, p = _case("shell")
    b = _case("shell")[0]
    for g in (a, b):
        g.init_run()
        g.run(5)
    h = a.get_state(HF)
    s = b.get_state(gamhip.GAM_OSTATE)
    s["Gas"][...] *= 1.5
    if after == "init":
        b.init_run()
    elif after == "put_old":
        b.put_state(s, gamhip.GAM_OSTATE)
    elif after == "put_new":
        b.put_state(s)
        b.init_run()
    elif after == "bcs":
        b.enforce_bcs()
        b.bflux2fld()
        b.bflux2fld(gamhip.GAM_OSTATE)
    elif after == "grid":
        b.grid_from_corners(grid["xyz"])
    elif after == "init_step":
        # the half state is the new step's, whose oState is State
        a.init_run()
        b.init_run()
        a.step()
        b.run(1)
        h = a.get_state(HF)
    else:
        b.autotune(reps=1)
        # of a tuning step: the next step's
        a.step()
        h2, t = b.get_state(HF), a.get_state(HF)
        assert _worst(h2, t) <= TOL
        a.close()
        b.close()
        return
    h2 = b.get_state(HF)
    for k in KEYS:
        assert np.array_equal(h[k], h2[k]), k
    a.close()
    b.close()


@pytest.mark.parametrize("kind", ["box7", "shell", "hydro7"])
def test_states_put_between_steps_match_oracle(kind):
    """A state put after plain steps takes the predictor again: its density
    may lie below the floor and its ghost cells be anything.  Without a
    magnetic field the steps themselves leave densities below the floor."""
    g, o, grid, st, p = _case(kind, dFloor=0.95)
    g.init_run()
    o.init_run()
    g.run(3)
    for _ in range(3):
        o.step()
    o.st["Gas"][4:8, 4:8, 4:8, 0] *= 0.9
    o.st["Bxyz"][...] *= 1.01
    g.put_state({k: o.st[k] for k in KEYS} | {"time": g.get_state()["time"]})
    for q in range(4):
        g.step()
        o.step()
        assert max(compare_state(g, o).values()) <= TOL, q
    g.enforce_bcs()
    o.enforce_bcs()
    g.run(4)
    for _ in range(4):
        o.step()
    assert max(compare_state(g, o).values()) <= TOL
    g.close()
