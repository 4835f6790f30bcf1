"""The limiter of the reconstructions (pdm_lr in mage_amd/csrc/gam_phys.h),
compiled for the host, against the oracle's statement of PDM and pdmLR
(recon.F90:231-301) over every 4-tuple of limiter values in {-2 .. 2, NaN}
and values below, inside and above them, NaN too.

Equal to 4 ulp of the largest value where the oracle's pair is finite; NaN
in the pair (a face's flux takes both sides) exactly where the oracle has
it: a broken cell is not hidden from the faces whose limiter it enters.
"""
import ctypes as C
import itertools
import os
import subprocess

import numpy as np
import pytest

import pyoracle as po

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r'''
#include "gam_phys.h"
extern "C" void pdm(int n, double b, const double *q, const double *l, const double *r, double *ql, double *qr)
{ for (int i = 0; i < n; i++) pdm_lr(b, q + 4 * i, l[i], r[i], ql[i], qr[i]); }
'''
DP = C.POINTER(C.c_double)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("limiter")
    (d / "pdm_host.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-std=c++17",
                    "-I", os.path.join(ROOT, "tests", "host_shim"), "-I", os.path.join(ROOT, "mage_amd", "csrc"),
                    str(d / "pdm_host.cpp"), "-o", str(d / "libpdm.so")], check=True)
    L = C.CDLL(str(d / "libpdm.so"))
    L.pdm.argtypes = [C.c_int, C.c_double, DP, DP, DP, DP, DP]
    return L


@pytest.mark.parametrize("form", ["pair", "single"])
@pytest.mark.parametrize("b", [0.75, 1e6])
def test_limiter_matches_oracle_nan_included(lib, b, form):
    O = po.lib()
    O.orc_pdm.restype = C.c_double
    O.orc_pdm.argtypes = [C.c_double] * 5
    O.orc_pdm_lr.argtypes = [C.c_double, DP, C.c_double, DP, DP]
    nan = float("nan")
    v = (-2.0, -1.0, 0.0, 1.0, 2.0, nan)
    lr = [(-3.0, -3.0), (-0.4, -0.4), (0.0, 0.0), (1.3, 1.3), (3.0, 3.0), (nan, nan)]
    if form == "single":     # the two sides' own values (7UP)
        lr = [(-0.4, 1.3), (3.0, -3.0), (nan, 0.5), (0.5, nan)]
    cases = list(itertools.product(itertools.product(v, repeat=4), lr))
    q = np.array([c[0] for c in cases]).ravel()
    l = np.array([c[1][0] for c in cases])
    r = np.array([c[1][1] for c in cases])
    ql, qr = np.empty(len(l)), np.empty(len(l))
    lib.pdm(len(l), b, *[a.ctypes.data_as(DP) for a in (q, l, r, ql, qr)])
    for n, (t, (x, y)) in enumerate(cases):
        if form == "pair":
            a = (C.c_double * 4)(*t)
            cl, cr = C.c_double(), C.c_double()
            O.orc_pdm_lr(b, a, x, C.byref(cl), C.byref(cr))
            want = cl.value, cr.value
        else:
            want = O.orc_pdm(b, t[0], t[1], t[2], x), O.orc_pdm(b, t[3], t[2], t[1], y)
        assert np.isnan(ql[n] + qr[n]) == np.isnan(want[0] + want[1]), (t, x, y)
        if np.isfinite(want[0] + want[1]):
            assert abs(ql[n] - want[0]) <= 4 * 2.3e-16 * 3 and abs(qr[n] - want[1]) <= 4 * 2.3e-16 * 3, (t, x, y)
