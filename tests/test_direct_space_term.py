"""The FP64 pair kernel's direct-space term, evaluated as the kernel does (every
operation rounded to double, fused multiply-adds once), against 60 digits (CPU).

Bounds, on the RMS relative error in each range of r: half-ulp roundings are
0.42e-16 RMS of their result on average.  The force factor goes through ten of them
(1/r, 1/r^2, 1/r^3 with 1/r's own, the polynomial's last, q, the scaled product,
the product with 1/r^3) and 0.7e-16 of truncation: 2.1e-16.  The energy through
five, and the truncation counts against E, which falls to a fifth: 3.5e-16.  Beside
that, no range may be worse than the formula with library functions that round
correctly, by more than a tenth for the force (1.9e-16 to 7.7e-16).
"""
import os
import re

import numpy as np
import pytest

mp = pytest.importorskip("mpmath")

SRC = open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "nexusmd_amd", "csrc", "nx_device.h")).read()
RANGES = [(0.1, 0.2), (0.2, 0.3), (0.3, 0.45), (0.45, 0.65), (0.65, 0.85), (0.85, 1.0)]


def _coefficients(name):
    text = re.search(name + r"\[\d+\] = \{(.*?)\};", SRC, re.S).group(1)
    return [mp.mpf(float(v)) for v in text.replace("\n", " ").split(",") if v.strip()]


def _rnd(v):
    return mp.mpf(float(v))


def _fma(a, b, c):
    return _rnd(a * b + c)


def _kernel(r2, alpha, kerfcx, kexp2m1, seed_error):
    ex = alpha * alpha / mp.log(2)
    ew_exp = _rnd(ex)
    ew_lo, ew_u, ew_q = _rnd(ex - ew_exp), _rnd(alpha / mp.sqrt(2)), _rnd(2 * alpha / mp.sqrt(mp.pi))
    y = _rnd((1 + seed_error) / mp.sqrt(r2))
    err = _fma(-_rnd(r2 * y), y, 1)
    y = _fma(_rnd(y * err), _fma(mp.mpf(0.375), err, mp.mpf(0.5)), y)
    y2 = _rnd(y * y)
    y2 = _fma(y2, _fma(-r2, y2, 1), y2)
    r = _rnd(r2 * y)
    magic = mp.mpf(6755399441055744)
    big = _fma(r2, -ew_exp, magic)
    f = _fma(r2, -ew_lo, _fma(r2, -ew_exp, -(big - magic)))
    u = _fma(r, ew_u, -1)
    u2 = _rnd(u * u)
    p, o, e = kexp2m1[10], kerfcx[23], kerfcx[24]
    for k in range(11, -1, -1):
        e = _fma(e, u2, kerfcx[2 * k])
        if k > 0:
            o = _fma(o, u2, kerfcx[2 * k - 1])
        if k < 10:
            p = _fma(p, f, kexp2m1[k])
    e = _fma(o, u, e)
    fp = _rnd(p * f)
    q = _fma(r, ew_q, e)
    scale = mp.mpf(2) ** int(big - magic)
    return (_rnd(_fma(fp, q, q) * scale * _rnd(y2 * y)), _rnd(_fma(fp, e, e) * scale * y))


def _library(r2, alpha):
    r = _rnd(mp.sqrt(r2))
    ir, ar = _rnd(1 / r), _rnd(alpha * r)
    c, x = _rnd(mp.erfc(ar)), _rnd(mp.exp(_rnd(-ar * ar)))
    t = _rnd(c + _rnd(_rnd(_rnd(2 * ar) * x) / _rnd(mp.sqrt(mp.pi))))
    return _rnd(_rnd(_rnd(ir * ir) * ir) * t), _rnd(ir * c)


@pytest.mark.parametrize("tol", [5e-4, 1.7e-4])      # the second: alpha^2 rc^2 = 7.99, the end of the range
def test_direct_space_term_against_60_digits(tol):
    with mp.workdps(60):
        kerfcx, kexp2m1 = _coefficients("kErfcx"), _coefficients("kExp2m1")
        assert len(kerfcx) == 25 and len(kexp2m1) == 11
        alpha = _rnd(mp.sqrt(-mp.log(2 * mp.mpf(tol))))
        rng = np.random.default_rng(5)
        for lo, hi in RANGES:
            rel = []
            for r in rng.uniform(lo, hi, 150):
                r2 = mp.mpf(float(r * r))
                x = alpha * mp.sqrt(r2)
                exact = ((mp.erfc(x) + 2 * x * mp.exp(-x * x) / mp.sqrt(mp.pi)) / mp.sqrt(r2) ** 3, mp.erfc(x) / mp.sqrt(r2))
                seed = mp.mpf(float(rng.uniform(-1, 1))) * mp.mpf(2) ** -26
                got = _kernel(r2, alpha, kerfcx, kexp2m1, seed) + _library(r2, alpha)
                rel.append([float(abs(g / exact[k % 2] - 1)) for k, g in enumerate(got)])
            force, energy, force_lib, _ = np.sqrt((np.array(rel) ** 2).mean(0))
            print("r %.2f-%.2f: force %.2e (library %.2e), energy %.2e" % (lo, hi, force, force_lib, energy))
            assert force <= 2.1e-16 and energy <= 3.5e-16
            assert force <= 1.1 * force_lib


def test_energy_factor_of_a_close_pair():
    """erfc(alpha r) / r and the force factor at r -> 0: 1 / r and 1 / r^3 to rounding."""
    with mp.workdps(60):
        kerfcx, kexp2m1 = _coefficients("kErfcx"), _coefficients("kExp2m1")
        alpha = _rnd(mp.mpf(2.6))
        for r in (1e-4, 1e-3, 0.02):
            r2 = mp.mpf(float(r * r))
            f, e = _kernel(r2, alpha, kerfcx, kexp2m1, mp.mpf(0))
            x = alpha * mp.sqrt(r2)
            assert abs(e * mp.sqrt(r2) / mp.erfc(x) - 1) < 1e-15
            assert abs(f * mp.sqrt(r2) ** 3 / (mp.erfc(x) + 2 * x * mp.exp(-x * x) / mp.sqrt(mp.pi)) - 1) < 1e-15
