"""State arrays in device memory of the context's GPU (torch tensors) and in
pinned host memory, in and out, for State, oState and the half state, whose
Efld is zero wherever the array lies: equal to the same calls with pageable
host arrays."""
import ctypes as C

import numpy as np
import pytest
import torch

from helpers import box_case, shell_case
from mage_amd import gamhip

pytestmark = pytest.mark.gpu
KEYS = ("Gas", "magFlux", "Bxyz", "Efld")


def _tensors(g, kind, fill):
    c = g.Ni * g.Nj * g.Nk
    f = (g.Ni + 1) * (g.Nj + 1) * (g.Nk + 1)
    kw = {"device": "cuda:0"} if kind == "device" else {"pin_memory": True}
    return {k: torch.full((n,), fill, dtype=torch.float64, **kw)
            for k, n in (("Gas", 5 * c), ("magFlux", 3 * f), ("Bxyz", 3 * c), ("Efld", 3 * c))}


def _args(t):
    return [C.cast(t[k].data_ptr(), gamhip.DP) for k in KEYS]


@pytest.mark.parametrize("kind", ["device", "pinned"])
@pytest.mark.parametrize("which", [gamhip.GAM_STATE, gamhip.GAM_OSTATE, gamhip.GAM_HFSTATE])
@pytest.mark.parametrize("case", ["box", "shell"])
def test_states_in_device_and_pinned_memory(case, which, kind):
    mk = lambda: shell_case((16, 11, 13), state="mhd")[0] if case == "shell" else box_case((16, 9, 11))[0]
    g = mk()
    g.init_run()
    g.run(3)
    want = g.get_state(which)
    t = _tensors(g, kind, 7.0)
    torch.cuda.synchronize()
    time = C.c_double()
    g._chk(g.L.gam_get_state(g.ctx, which, *_args(t), C.byref(time)))
    assert time.value == want["time"]
    for k in KEYS:
        a = t[k].cpu().numpy().reshape(want[k].shape, order="F")
        assert np.array_equal(a, want[k]), k
    if which != gamhip.GAM_HFSTATE:
        h = mk()
        h.init_run()
        h._chk(h.L.gam_put_state(h.ctx, which, *_args(t), time.value))
        back = h.get_state(which)
        for k in KEYS:
            assert np.array_equal(back[k], want[k]), k
        h.close()
    else:
        assert not np.any(want["Efld"])
    g.close()
