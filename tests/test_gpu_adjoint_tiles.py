"""The adjoint's tiles against translation of the problem.

On the periodic box a state, objective weights and all moved by s cells
along an axis must give the gradient moved by s cells: every face and edge
then lies at another place of its tile, so sums at a tile's ends, remainders
of 1 to 15 and rows cut anywhere along i show against the same sums inside a
tile.  (That the gradient itself is right is the finite-difference tests'
part.)

The two runs see corner coordinates that differ in the last place, so
metrics differ by ~1e-15 / dx relative, ~1e-14; the step and its
transpose amplify that by the stencils' weights and the divisions by
cell volumes, at most ~100.  Bar: 1e-10 of the largest gradient entry of
the same variable.  Every variable varies smoothly, so no limiter
difference is exactly 0.  One step: CalcDT reads one layer of ghost cells
before the boundary pass, so dt itself moves with the problem only at first.
"""
import numpy as np
import pytest

from helpers import box_case
from mage_amd import gamhip

pytestmark = pytest.mark.gpu


def _moved(a, N, s):
    """a with its interior moved by s cells (ghosts and last faces follow)."""
    for ax in range(3):
        q = (np.arange(a.shape[ax]) - 4 - s[ax]) % N[ax] + 4
        a = np.take(a, q, axis=ax)
    return np.asfortranarray(a)


def _wave(shape, N, c, ph):
    x = [2 * np.pi * (np.arange(n) - 4 + 0.5) / m for n, m in zip(shape, N)]
    return (np.sin(x[0] + ph)[:, None, None] * np.cos(x[1] - ph)[None, :, None]
            + 0.5 * np.sin(c * x[2] + 2 * ph)[None, None, :])


def _gradient(N, rmeth, s):
    g, o, grid, st, _ = box_case(N, rmeth)
    st = {k: st[k].copy(order="F") for k in ("Gas", "magFlux", "Bxyz", "Efld")}
    for v, amp in ((0, 0.05), (1, 0.02), (2, 0.03), (3, 0.02), (4, 0.06)):
        st["Gas"][..., v] += amp * np.max(np.abs(st["Gas"][..., v])) * _wave(st["Gas"].shape[:3], N, 1 + v % 2, 0.3 + v)
    w = 1.0 + 0.3 * _wave(grid["volume"].shape, N, 1, 0.7)
    w = _moved(w * np.mean(grid["volume"][4:-4, 4:-4, 4:-4]), N, s)
    for ax in range(3):   # (the objective sums over the ghosts too)
        q = [slice(None)] * 3
        for q[ax] in (slice(0, 4), slice(4 + N[ax], None)):
            w[tuple(q)] = 0.0
    g.put_state({k: _moved(a, N, s) for k, a in st.items()})
    g.init_run()
    adj = gamhip.GamAdjoint(g, 1, 1)
    adj.set_weights(w)
    adj.forward()
    out = adj.backward(fluxes=True)
    adj.close()
    g.close()
    inner = tuple(slice(4, 4 + n) for n in N)
    res = []
    for q, a in enumerate(out):
        a = a.copy()
        if q >= 2:
            for ax in range(3):   # a direction's last face is its first one
                lo, hi = [slice(None)] * 3 + [ax], [slice(None)] * 3 + [ax]
                lo[ax], hi[ax] = 4, 4 + N[ax]
                a[tuple(lo)] += a[tuple(hi)]
        res.append(a[inner])
    return res


@pytest.mark.parametrize("N,s", [((16, 8, 9), (3, 1, 4)), ((24, 15, 16), (11, 6, 9)),
                                 ((40, 17, 31), (7, 16, 15)), ((32, 33, 8), (16, 1, 5))])
@pytest.mark.parametrize("rmeth", ["8CENT", "7UP"])
def test_gradient_moves_with_the_problem(rmeth, N, s):
    print("adjoint of the %s %s box moved by %s" % (N, rmeth, s), flush=True)
    a, b = _gradient(N, rmeth, (0, 0, 0)), _gradient(N, rmeth, s)
    for q, (x, y) in enumerate(zip(a, b)):
        x = np.roll(x, s, axis=(0, 1, 2))
        for v in range(x.shape[3]):
            err, big = np.max(np.abs(x[..., v] - y[..., v])), np.max(np.abs(x[..., v]))
            assert big > 0.0 and err <= 1e-10 * big, (q, v, err, big)
