"""Grids large enough that the fluxes and EMFs of the three directions take
turns in slabs along k, against one launch per direction (which has no
slabs): extents that leave remainders in every tile and slab, and slab
counts limited by the extent along k and by the chunks.

Same kernels' arithmetic but for products the compiler contracts
differently: 1e-12 relative L-infinity after 3 steps, as in
test_gpu_step.py.
"""
import numpy as np
import pytest

from helpers import rel_linf, shell_case
from mage_amd import gamhip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [(104, 75, 91), (96, 9, 641), (208, 301, 9)])
def test_slabs_match_single_direction_launches(N):
    print("slabs on the %s shell" % (N,), flush=True)
    out = []
    for apart in (False, True):
        g, o, grid, st, p = shell_case(N, state="mhd")
        if apart:
            plan = g.get_plan()
            plan["emf_i"] = 9          # direct loads: nothing is merged
            g.set_plan(plan)
        g.init_run()
        g.run(3)
        out.append(g.get_state())
        out[-1]["hf"] = g.get_state(gamhip.GAM_HFSTATE)["Gas"]
        g.close()
    for k in ("Gas", "magFlux", "Bxyz", "Efld", "hf"):
        assert np.all(np.isfinite(out[0][k]))
        assert rel_linf(out[0][k], out[1][k]) <= 1e-12, k
