"""gam_erfc_exp of a NaN is NaN in both results, as erfc's and exp's are
(stress.F90:474-475): a broken face state shows in every flux it enters."""
import ctypes as C
import os
import subprocess

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_erfc_of_nan_is_nan(tmp_path):
    src, so = tmp_path / "e.cpp", tmp_path / "libe.so"
    src.write_text('#include "gam_erfc.h"\n'
                   'extern "C" double eval(double z, double *e) { return gam_erfc_exp(z, *e); }\n')
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-std=c++17",
                    "-I", os.path.join(ROOT, "mage_amd", "csrc"), str(src), "-o", str(so)], check=True)
    f = C.CDLL(str(so)).eval
    f.restype, f.argtypes = C.c_double, [C.c_double, C.POINTER(C.c_double)]
    for z in (float("nan"), -float("nan")):
        e = C.c_double()
        assert np.isnan(f(z, C.byref(e))) and np.isnan(e.value)
