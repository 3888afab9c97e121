"""An FP64 request's trajectory is the same bits alone and beside systems that
make its batch take other kernels: the terms in launches of their own (by the
batch's atoms), the pair kernel that chooses the direct space per system, line
passes instead of planes."""
import numpy as np
import pytest

from nexusmd_amd import _lib as L
from nexusmd_amd import engine as E
from nexusmd_amd import systems as S

from _util import bare_system

pytestmark = pytest.mark.gpu

DT = 0.0005


def _request():
    s = S.bead_chain(n=400, L=2.6, grid=(24, 24, 24), seed=11)
    s.pos = (s.pos + np.random.default_rng(1).normal(0.0, 0.004, s.pos.shape)) % s.L
    s.vel = S.maxwell_boltzmann(s.mass, 300.0, np.random.default_rng(2))
    return s


def _small(tol=5e-4, grid=(24, 24, 24)):
    rng = np.random.default_rng(3)
    g = np.stack(np.meshgrid(*[np.arange(8) + 0.5] * 3, indexing="ij"), -1).reshape(-1, 3) * (2.4 / 8)
    q = rng.normal(0.0, 0.3, len(g))
    s = bare_system(g, np.zeros(3), np.full(3, 2.4), q=q - q.mean(), sig=np.full(len(g), 0.15),
                    eps=np.full(len(g), 0.2), mass=np.full(len(g), 16.0), grid=grid, ewald_tol=tol)
    return s


def _run(systems, prec):
    srv = E.Server(precision=prec, budget_bytes=32 << 30, max_active=8)
    ids = [srv.submit(s, 12, DT) for s in systems]
    srv.run()
    assert [srv.poll(i)[0] for i in ids] == [2] * len(ids)
    p, v, e = srv.fetch(ids[0])
    srv.close()
    return p, v, e


@pytest.mark.parametrize("beside", ["60,000 atoms", "a tight tolerance", "a grid in lines"])
def test_fp64_request_alone_and_beside(beside):
    if beside == "60,000 atoms":
        other = S.water_box(n_mol=20000, L=8.44, grid=(80, 80, 80), seed=5)
    elif beside == "a tight tolerance":
        other = _small(tol=1e-6)
    else:
        other = _small(grid=(24, 150, 100))
    print("[gpu] FP64 request beside %s" % beside, flush=True)
    p0, v0, e0 = _run([_request()], L.FP64)
    p1, v1, e1 = _run([_request(), other], L.FP64)
    np.testing.assert_array_equal(p1, p0)
    np.testing.assert_array_equal(v1, v0)
    assert e1 == e0
