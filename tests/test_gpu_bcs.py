"""Boundary conditions by look-up against the oracle's side-by-side passes:
every grouping of axes into launches (all periodic; i apart; j apart) and
mixed kinds of the two sides of an axis, on extents that are not multiples
of a tile.  Whole arrays, ghost cells and outermost faces included.

Tolerances (relative L-infinity): 1e-13 for copies (the outer zero gradient
of i computes), 1e-12 after two steps, as in test_gpu_step.py.
"""
import numpy as np
import pytest

from helpers import box_case, compare_state, shell_case

pytestmark = pytest.mark.gpu

P, Z = "periodic", "zerograd"
BOX = [
    [P, P, P, P, P, P],
    [P, P, Z, Z, P, P],
    [P, P, P, P, Z, Z],
    [Z, Z, P, P, P, P],
    [Z, Z, P, P, Z, Z],
    [Z, Z, Z, Z, Z, Z],
    [P, Z, Z, P, P, P],
    [Z, P, P, Z, Z, P],
    ["sphin", "sphout", Z, Z, P, P],
    ["sphin", Z, P, P, Z, Z],
    [P, "sphout", P, P, P, P],
]


@pytest.mark.parametrize("bcs", BOX, ids=lambda b: "-".join(x[:4] for x in b))
def test_enforce_bcs_and_steps_match_oracle(bcs):
    N = (16, 9, 11)
    g, o, grid, st, p = box_case(N, "7UP", bc=bcs)
    rng = np.random.default_rng(11)
    for k in ("Gas", "magFlux", "Bxyz"):
        a = o.st[k]
        a[...] = rng.standard_normal(a.shape)
    o.st["Gas"][..., 0] = np.abs(o.st["Gas"][..., 0]) + 1.0
    g.put_state({k: o.st[k] for k in ("Gas", "magFlux", "Bxyz", "Efld")})
    g.enforce_bcs()
    o.enforce_bcs()
    e = compare_state(g, o, ("Gas", "magFlux", "Bxyz"))
    assert max(e.values()) <= 1e-13, e
    g.close()

    g, o, grid, st, p = box_case(N, "7UP", bc=bcs)
    g.init_run()
    o.init_run()
    for _ in range(2):
        g.step()
        o.step()
    e = compare_state(g, o)
    assert max(e.values()) <= 1e-12, e
    g.close()


@pytest.mark.parametrize("k", [P, Z])
@pytest.mark.parametrize("outi", ["wind", "sphout"])
def test_shell_walls_match_oracle(outi, k):
    g, o, grid, st, p = shell_case((16, 11, 13), state="mhd", bc=[Z, outi, Z, Z, k, k])
    g.init_run()
    o.init_run()
    for _ in range(2):
        g.step()
        o.step()
    e = compare_state(g, o)
    assert max(e.values()) <= 1e-12, e
    g.close()
