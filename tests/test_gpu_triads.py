"""Interface fluxes with and without the shortened form for orthonormal face
triads (the tangential velocity as what the normal leaves of it): grids
whose uploaded triads are orthonormal to rounding take it, others the
general form.  Both against the oracle on the same metrics: relative
L-infinity 1e-12 after one step, as in test_gpu_step.py.
"""
import numpy as np
import pytest

import pyoracle as po
from helpers import compare_state, shell_case
from mage_amd import gamhip, problems as pb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rmeth", ["7UP", "8CENT"])
@pytest.mark.parametrize("tilt", [0.0, 1e-13, 0.05])
def test_uploaded_triads_match_oracle(tilt, rmeth):
    """tilt: each T1 leans towards T2 by this much (0: orthonormal)."""
    g0, o0, grid, st, p = shell_case((16, 11, 13), rmeth, state="mhd")
    g0.close()
    Tf = grid["Tf"]
    Tf[..., 3:6, :] += tilt * Tf[..., 6:9, :]
    wind = pb.constant_wind()
    g = gamhip.GamHip(16, 11, 13, p)
    g.set_grid(grid)
    g.set_background(grid)
    g.set_wind(wind)
    o = po.Oracle(16, 11, 13, p, grid, wind=wind)
    g.put_state(st)
    o.set_state(st)
    g.init_run()
    o.init_run()
    g.step()
    o.step()
    e = compare_state(g, o)
    assert max(e.values()) <= 1e-12, e
    g.close()
