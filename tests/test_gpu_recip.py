"""The engine's own charge spread, transforms and convolution, by themselves.

A dozen charges farther apart than the cutoff feel the reciprocal sum alone, so
forces and energy test the path a step takes (the spread inside the forward
pass, the product inside the x pass), not the standalone transforms'.  Against
the FP64 oracle: forces 1e-9 relative RMS and energies 1e-9 in FP64, 5e-4 and
1e-5 in the mixed path (the bounds of the other parity tests).
"""
import numpy as np
import pytest

from nexusmd_amd import _lib as L
from nexusmd_amd import engine as E
from oracle import pyoracle as O

from _util import bare_system, rel_rms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("passes", ["plane", "lines"])
@pytest.mark.parametrize("grid", [(30, 36, 25), (8, 27, 64), (100, 15, 24), (24, 125, 9)])
def test_reciprocal_sum_alone(grid, passes, prec, monkeypatch):
    monkeypatch.setenv("NEXUSMD_FFT_PLANE", "1" if passes == "plane" else "0")
    rng = np.random.default_rng(7)
    box = np.array([2.0, 2.0, 3.0])
    g = np.stack(np.meshgrid(np.arange(2), np.arange(2), np.arange(3), indexing="ij"), -1).reshape(-1, 3)
    pos = (g + 0.25 + rng.uniform(-0.1, 0.1, g.shape)) * [1.0, 1.0, 1.0]
    q = rng.normal(0.0, 0.7, len(pos))
    s = bare_system(pos, np.zeros(3), box, q=q - q.mean(), cutoff=0.75, grid=grid)
    print("[gpu] reciprocal sum %s %s precision %d" % (grid, passes, prec), flush=True)
    ctx = E.Context(s, precision=prec)
    f, e = ctx.compute_forces()
    ctx.close()
    ref, er = O.compute_forces(O.Prepared(s))
    assert e["coulomb_direct"] == 0.0 and er["coulomb"] == 0.0
    assert rel_rms(f, ref) <= (1e-9 if prec == L.FP64 else 5e-4)
    assert abs(e["recip"] - er["recip"]) <= (1e-9 if prec == L.FP64 else 1e-5) * abs(er["recip"])
