"""Coefficients of the FP64 direct-space series (csrc/nx_device.h)."""
import os
import re

import numpy as np
import pytest


def test_erf_series_against_mpmath():
    """The coefficients of the series, evaluated as the kernel does, against 30
    digits: absolute error below 2e-16 (half an ulp of their sum, 1.13 and 0.75,
    for the last addition and as much again for the rest)."""
    mp = pytest.importorskip("mpmath")
    mp.mp.dps = 30
    src = open(os.path.join(os.path.dirname(__file__), "..", "nexusmd_amd", "csrc", "nx_device.h")).read()
    for name, f in (("kErfA", lambda x: mp.erf(x) / x),
                    ("kErfB", lambda x: (mp.erf(x) - 2 * x * mp.exp(-x * x) / mp.sqrt(mp.pi)) / x ** 3)):
        c = [float(v) for v in re.search(name + r"\[\d+\] = \{(.*?)\};", src, re.S).group(1).replace("\n", " ").split(",") if v.strip()]
        for s in np.linspace(0.004, 8.0, 61):
            u = s * 0.25 - 1.0
            got = float(np.polynomial.polynomial.polyval(u, c))
            assert abs(got - float(f(mp.sqrt(mp.mpf(float(s)))))) < 2e-16 * (1.13 if name == "kErfA" else 1.0), (name, s)
