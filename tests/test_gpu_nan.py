"""A broken cell (NaN momentum) or face (NaN magnetic flux) reaches the same
cells and faces as in the oracle, step by step: through the predictor (the
first two steps of a state that was put) and without it.  Every kernel that
drops or keeps a NaN shows in the masks, which are compared exactly.
"""
import numpy as np
import pytest

from helpers import box_case, shell_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rmeth", ["8CENT", "7UP"])
@pytest.mark.parametrize("what,kind", [("cell", "box"), ("cell", "hydro"), ("cell", "shell"), ("face", "box"),
                                       ("face", "shell")])
def test_nan_spreads_as_in_the_oracle(what, kind, rmeth):
    N = (32, 27, 29)
    if kind == "shell":
        g, o, grid, st, p = shell_case(N, rmeth, state="mhd")
    else:
        g, o, grid, st, p = box_case(N, rmeth, doMHD=0 if kind == "hydro" else 1)
    g.init_run()
    o.init_run()
    for s in (o.st, o.ost):
        if what == "cell":
            s["Gas"][18, 17, 19, 1] = np.nan
        else:
            s["magFlux"][18, 17, 19, 0] = np.nan
    for which, s in ((0, o.st), (1, o.ost)):
        t = g.get_state(which)["time"]
        g.put_state({"Gas": s["Gas"], "magFlux": s["magFlux"], "time": t}, which)
    n = 0
    for q in range(3):
        g.step(sync=False)      # (CalcDT is not the matter here)
        o.step()
        a = g.get_state()
        for k in ("Gas", "magFlux", "Efld"):
            x, y = np.isnan(a[k]), np.isnan(o.st[k])
            if k != "Efld":
                x, y = (z[4:4 + N[0], 4:4 + N[1], 4:4 + N[2]] for z in (x, y))
            assert np.array_equal(x, y), (q, k, int(x.sum()), int(y.sum()), int((x & ~y).sum()))
        n = int(np.isnan(a["Gas"]).sum())
    assert n > 0
    g.close()
