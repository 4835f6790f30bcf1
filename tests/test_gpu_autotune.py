"""gam_autotune from plans with a slow choice: it keeps a better update shape
whatever the flux and EMF slots' own launches measure, and finds its way from
direct loads in every flux and EMF slot to the forms that need no predictor.
State, time and dt are left as they were.

The slow choices cost 6 % (the update) and 20 % of a step of this shell;
autotune acts on 1 %.
"""
import numpy as np
import pytest

from helpers import shell_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slow", ["update", "direct"])
def test_autotune_replaces_slow_choices(slow):
    g = shell_case((48, 48, 64), state="mhd")[0]
    plan = dict(g.get_plan())
    lds = {k: v for k, v in plan.items() if k[:3] in ("emf", "flu")}
    if slow == "update":
        plan["update"] = 18
    else:
        plan.update({k: 9 for k in lds})
    g.set_plan(plan)
    g.init_run()
    g.run(4)
    t0, s0 = g.get_time(), g.get_state()
    tuned = g.autotune(reps=8)
    print("tuned plan", tuned, flush=True)
    assert g.get_time() == t0
    s1 = g.get_state()
    assert all(np.array_equal(s0[k], s1[k]) for k in ("Gas", "magFlux", "Bxyz", "Efld"))
    if slow == "update":
        assert tuned["update"] != 18
    # no slot back at direct loads: values of the LDS forms
    for k in lds:
        assert tuned[k] in ((1, 2, 3) if k[:3] == "emf" else (1, 2) if k == "flux_i" else (4, 5, 6, 7)), k
    g.close()
