"""Contexts without room for the primitives beside their states (forced by
GAM_MEM_LIMIT, which gam_create takes for a full device): 208 planes of rows
of Nip + 16, the memory such a context needs at all, and the results of any
other context.

Steps against the oracle: 1e-12 relative L-infinity, as in test_gpu_step.py.
The adjoint runs the same kernels on either layout: 1e-12.
"""
import numpy as np
import pytest

from helpers import box_case, compare_state, rel_linf, shell_case
from hip_runtime import used
from mage_amd import gamhip, problems as pb

pytestmark = pytest.mark.gpu


def _planes(N, n):
    """Bytes of n planes of 64-byte rows."""
    pts = (N[0] + 16) * (N[1] + 9) * (N[2] + 9)
    return n * 8 * ((pts + 63) // 64 * 64)


def test_footprint_and_refusal(monkeypatch):
    N = (104, 96, 96)
    p = pb.shell_params("7UP")
    gamhip.GamHip(16, 8, 8, p).close()      # modules and the runtime's own memory
    need = _planes(N, 208)
    slack = 48 << 20                        # allocation granularity
    for limit in (None, need, need - 1):
        if limit is not None:
            monkeypatch.setenv("GAM_MEM_LIMIT", str(limit))
        u0 = used()
        if limit == need - 1:
            with pytest.raises(gamhip.GamError) as ei:
                gamhip.GamHip(*N, p)
            assert ei.value.code == -2      # GAM_E_HIP, as on a full device
            assert used() - u0 <= slack
            continue
        g = gamhip.GamHip(*N, p)
        mem = used() - u0
        print("limit %s: %.1f MiB" % (limit, mem / 2 ** 20), flush=True)
        if limit is None:
            assert mem >= _planes(N, 218)
        else:
            assert mem <= need + slack
        g.close()
        assert used() - u0 <= slack


def _case(kind, rmeth):
    if kind == "shell":
        return shell_case((24, 11, 13), rmeth, state="mhd")
    return box_case((24, 9, 11), rmeth, doMHD=0 if kind == "hydro" else 1)


@pytest.mark.parametrize("rmeth", ["8CENT", "7UP"])
@pytest.mark.parametrize("kind", ["box", "hydro", "shell"])
def test_results_without_room(kind, rmeth, monkeypatch):
    N = (24, 9, 11) if kind != "shell" else (24, 11, 13)
    full = _case(kind, rmeth)[0]
    monkeypatch.setenv("GAM_MEM_LIMIT", str(_planes(N, 208)))
    g, o, grid, st, p = _case(kind, rmeth)
    g.init_run()
    o.init_run()
    g.run(3)
    g.step()
    e = gamhip.GamEnsemble([g])
    e.run(2)
    e.close()
    g.enforce_bcs()
    g.run(2)
    for q in range(6):
        o.step()
    o.enforce_bcs()
    for q in range(2):
        o.step()
    assert max(compare_state(g, o).values()) <= 1e-12
    h, ho = g.get_state(gamhip.GAM_HFSTATE), o.half_state()
    assert max(rel_linf(h[k], ho[k]) for k in ("Gas", "magFlux", "Bxyz")) <= 1e-12
    d = g.divb()
    assert np.isfinite(d)
    monkeypatch.delenv("GAM_MEM_LIMIT")     # (it bounds a tuning run's snapshot too)
    g.autotune(reps=1)
    g.close()
    # the adjoint, against the context with every plane
    monkeypatch.setenv("GAM_MEM_LIMIT", str(_planes(N, 208)))
    g = _case(kind, rmeth)[0]
    grads = []
    for c in (full, g):
        c.init_run()
        a = gamhip.GamAdjoint(c, 3, 2)
        w = np.zeros(c.cshape, order="F")
        w[4:-4, 4:-4, 4:-4] = grid["volume"][4:-4, 4:-4, 4:-4]
        a.set_weights(w)
        J = a.forward()
        grads.append((J,) + a.backward(fluxes=kind != "hydro"))
        a.close()
        c.close()
    assert abs(grads[0][0] - grads[1][0]) <= 1e-12 * abs(grads[0][0])
    for x, y in zip(grads[0][1:], grads[1][1:]):
        assert rel_linf(x, y) <= 1e-12


def test_autotune_without_room_for_the_primitives(monkeypatch):
    """The snapshot of a tuning run takes the two states' 28 planes, with
    their primitives 38 where there is room: the run goes on within 1e-12
    (two steps through the predictor) or bit for bit."""
    N = (24, 11, 13)
    pts = ((24 + 9 + 15) // 16 * 16) * (N[1] + 9) * (N[2] + 9) + 16
    plane = 8 * ((pts + 63) // 64 * 64)
    ref = _case("shell", "7UP")[0]
    ref.init_run()
    ref.run(8)
    for planes, ok in ((218 + 38, True), (218 + 28, True), (218 + 27, False)):
        monkeypatch.delenv("GAM_MEM_LIMIT", raising=False)
        g = _case("shell", "7UP")[0]
        g.init_run()
        g.run(4)
        plan, s0, t0 = g.get_plan(), g.get_state(), g.get_time()
        monkeypatch.setenv("GAM_MEM_LIMIT", str(planes * plane))
        if ok:
            g.autotune(reps=1)
            g.set_plan(plan)
        else:
            with pytest.raises(gamhip.GamError) as ei:
                g.autotune(reps=1)
            assert ei.value.code == -2
        assert g.get_time() == t0
        s1 = g.get_state()
        for k in ("Gas", "magFlux", "Bxyz", "Efld"):
            assert np.array_equal(s0[k], s1[k])
        g.run(4)
        a, b = g.get_state(), ref.get_state()
        for k in ("Gas", "magFlux", "Bxyz", "Efld"):
            assert rel_linf(a[k], b[k]) <= (1e-12 if planes == 218 + 28 else 0.0), (planes, k)
        g.close()
    ref.close()
