"""The coefficients of the SE(3) exponential by their power series
(exp_series in yetanotherslam_amd/csrc/yas_tracker_dev.hpp), compiled for the
host here (hipcc), against exact rational sums: over the whole range that the
series is taken for, its ends included."""
import ctypes
import os
import shutil
import subprocess
from fractions import Fraction
from math import factorial

import numpy as np
import pytest

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
CSRC = os.path.join(os.path.dirname(__file__), "..", "yetanotherslam_amd", "csrc")
SRC = r'''
#include "yas_tracker_dev.hpp"
extern "C" double series(double th2, double* abc) {
  yas::exp_series(th2, abc[0], abc[1], abc[2]);
  return yas::kExpSeriesMax;
}
'''


def _exact(th2, first):
    t, s = Fraction(th2), Fraction(0)
    for k in range(14):
        s += (-t) ** k / factorial(2 * k + first)
    return s


def test_series_is_within_two_roundings(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    src, so = tmp_path / "s.hip", tmp_path / "s.so"
    src.write_text(SRC)
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "-std=c++17", "-O2", "-ffp-contract=off", "-shared",
                    "-fPIC", "-I", CSRC, "-I", os.path.join(CSRC, "..", "..", "include"), str(src), "-o", str(so)],
                   check=True, capture_output=True)
    f = ctypes.CDLL(str(so)).series
    f.restype = ctypes.c_double
    f.argtypes = [ctypes.c_double, ctypes.c_void_p]
    abc = np.zeros(3)
    top = f(0.0, abc.ctypes.data)
    assert top == 0.25 and abc[0] == 1.0 and abc[1] == 0.5 and abc[2] == 1.0 / 6.0
    worst = 0.0
    for th2 in [5e-324, 1e-300, 1e-16, 1e-8] + list(np.geomspace(1e-12, 0.25, 400)) + [np.nextafter(0.25, 0)]:
        f(float(th2), abc.ctypes.data)
        for got, first in zip(abc, (1, 2, 3)):
            want = _exact(float(th2), first)
            worst = max(worst, abs(float((Fraction(float(got)) - want) / want)))
    # the constant's rounding and the last step's, and 1/80 of the step's before
    assert worst <= 2.1 * 2.0 ** -53, worst
