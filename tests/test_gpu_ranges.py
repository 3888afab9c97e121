"""Kernels at the edges of the ranges their launch rules choose between.

Forces of both paths against the FP64 oracle, relative RMS: FP64 <= 1e-9, mixed
<= 5e-4 (the bounds of the other parity tests).
"""
import numpy as np
import pytest

from nexusmd_amd import _lib as L
from nexusmd_amd import engine as E
from nexusmd_amd import systems as S
from oracle import pyoracle as O

from _util import bare_system, rel_rms

pytestmark = pytest.mark.gpu

TOL = {L.FP64: 1e-9, L.MIXED: 5e-4}


def _gas(n, box, seed, grid=(0, 0, 0), cutoff=0.9):
    """n charged LJ particles on a jittered lattice in an oblong box."""
    rng = np.random.default_rng(seed)
    box = np.asarray(box, float)
    k = np.ceil(box * (n / box.prod()) ** (1 / 3)).astype(int)
    while k.prod() < n:
        k[np.argmin(k / box)] += 1
    g = np.stack(np.meshgrid(*[np.arange(m) + 0.5 for m in k], indexing="ij"), -1).reshape(-1, 3) * (box / k)
    g = g[rng.permutation(len(g))[:n]] + rng.normal(0.0, 0.01, (n, 3))
    q = rng.normal(0.0, 0.5, n)
    return bare_system(g % box, np.zeros(3), box, q=q - q.mean(), sig=rng.uniform(0.15, 0.2, n),
                       eps=rng.uniform(0.1, 0.6, n), cutoff=cutoff, grid=grid)


def _check(sys, prec, what, **kw):
    print("[gpu] %s n=%d precision=%d" % (what, sys.n, prec), flush=True)
    ctx = E.Context(sys, precision=prec, **kw)
    f, _ = ctx.compute_forces()
    ctx.close()
    ref, _ = O.compute_forces(O.Prepared(sys))
    assert rel_rms(f, ref) <= TOL[prec]


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("n", [5, 5999, 6000])
def test_chunk_sizes(n, prec):
    """Either side of the size where the FP64 pair kernel takes shorter chunks,
    and a system with far fewer chunks than wavefronts."""
    _check(_gas(n, (2.1, 4.3, 5.9), n, grid=(20, 40, 60)), prec, "chunk sizes")


@pytest.mark.parametrize("tol", [1.7e-4, 1.6e-4, 1e-7])
def test_fp64_direct_space_either_side_of_the_series(tol):
    """alpha^2 rc^2 just inside and outside the range of the FP64 pair kernel's
    series (8), and far outside."""
    s = _gas(900, (2.2, 2.0, 2.4), 3, grid=(24, 24, 24))
    s.ewald_tol = tol
    s.pos[1] = (s.pos[0] + [0.03, 0.02, 0.01]) % s.L       # a close contact
    assert (-np.log(2 * tol) <= 8.0) == (tol == 1.7e-4)
    _check(s, L.FP64, "series range")


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("grid,skin", [((20, 24, 30), 0.1),      # whole planes
                                       ((27, 45, 25), 0.0),      # odd rows, no buffer
                                       ((6, 10, 9), 0.3),        # stencils of most of the box
                                       ((24, 150, 100), 0.1),    # rows of planes (FP64), a y pass
                                       ((15, 135, 160), 0.1),    # rows of planes (both)
                                       ((8, 9, 1000), 0.1)])     # two rows at a time
def test_spread_shapes(grid, skin, prec):
    """Charge spreading over whole planes and over rows, forces on every atom."""
    s = _gas(1203, (2.0, 2.9, 2.3), 17, grid=grid)
    s.pos = (s.pos - s.pos[5] - 1e-9) % s.L       # one atom just inside the far corner
    s.pos = s.pos[np.random.default_rng(1).permutation(s.n)]
    _check(s, prec, "spread %s" % (grid,), skin=skin)


def test_spread_of_large_charges():
    """Charges past the bound of the short conversion to fixed point (8 e in FP64)."""
    s = _gas(700, (2.0, 2.0, 2.0), 4, grid=(24, 24, 24))
    s.q *= 30.0
    assert (np.abs(s.q) > 8).sum() > 100 and (np.abs(s.q) < 8).sum() > 100
    _check(s, L.FP64, "large charges")


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
def test_line_and_plane_passes_agree(prec, monkeypatch):
    s = _gas(1500, (2.4, 2.6, 2.2), 8, grid=(30, 36, 25))
    out = []
    for plane in ("1", "0"):
        monkeypatch.setenv("NEXUSMD_FFT_PLANE", plane)
        ctx = E.Context(s, precision=prec)
        out.append(ctx.compute_forces()[0])
        ctx.close()
    # the inverse transforms differ (one or two real lines at a time), the spread and
    # the forward ones do not: rounding only
    assert rel_rms(out[0], out[1]) <= (1e-13 if prec == L.FP64 else 1e-6)


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("n,box", [(63, (2.0, 2.0, 2.0)), (64, (2.0, 2.0, 2.0)), (65, (2.0, 2.0, 2.0)),
                                   (777, (2.0, 2.1, 9.0)),      # tall columns
                                   (777, (9.0, 2.1, 2.0)),      # one column across
                                   (2500, (2.3, 2.3, 2.3))])    # a dense box: many super-clusters a column
def test_super_cluster_shapes(n, box, prec):
    """Columns with no, one, a part of one and many super-clusters; the pair set
    bit for bit in FP64."""
    s = _gas(n, box, n + 1, grid=(24, 24, 48))
    _check(s, prec, "super-clusters", skin=0.1)
    if prec == L.FP64:
        ctx = E.Context(s, precision=prec, skin=0.1)
        got = ctx.neighbor_pairs()
        ctx.close()
        want = O.pairs(s, O.exclusions(s), method="brute")
        assert len(got) == len(want) and set(map(tuple, got.tolist())) == set(map(tuple, want.tolist()))


def test_coincident_columns_sort_by_atom():
    """Atoms with equal coordinates on every axis in turn (ties in every sort of
    the super-cluster splits) keep a deterministic list: two contexts, one set of bits."""
    s = _gas(600, (2.2, 2.2, 2.2), 9, grid=(24, 24, 24))
    s.pos[:200, 0] = 0.7
    s.pos[150:400, 1] = 1.1
    s.pos[300:, 2] = 0.4 + 1.4 * (np.arange(300) % 2)
    s.pos[:, 2] += 1e-3 * np.arange(600)       # no two atoms on one point
    s.pos %= s.L
    s.eps[:] = 0.0                              # close contacts: charges alone
    _check(s, L.FP64, "ties")
    f = []
    for _ in range(2):
        ctx = E.Context(s, precision=L.MIXED)
        f.append(ctx.compute_forces()[0])
        ctx.close()
    np.testing.assert_array_equal(f[0], f[1])


@pytest.mark.parametrize("n", [7, 45000])       # one thread and several in the copies
def test_state_and_results_round_trip(n):
    """State in, report out: every buffer whole, in the caller's order, on a second
    state in the same context too; what was not asked for is not written."""
    s = _gas(n, (2.0, 2.0, 2.0) if n < 100 else (7.0, 7.4, 7.8), 2, grid=(20, 20, 20) if n < 100 else (64, 64, 64))
    rng = np.random.default_rng(3)
    ctx = E.Context(s, precision=L.FP64)
    for k in range(2):
        pos = (s.pos + 0.3 * k) % s.L
        vel = rng.normal(size=(n, 3))
        ctx.set_state(pos, vel)
        p, v = ctx.get_state()
        np.testing.assert_array_equal(p, pos)
        np.testing.assert_array_equal(v, vel)
        f0, e0 = ctx.compute_forces()
        p, v, f, e = ctx.step_report(0.0005)
        np.testing.assert_array_equal(p, pos)
        np.testing.assert_array_equal(v, vel)
        np.testing.assert_array_equal(f, f0)
        assert e["potential"] == e0["potential"]
        p, v = ctx.get_state()
        np.testing.assert_allclose(v, vel + 0.0005 * f / s.mass[:, None], rtol=1e-14, atol=1e-13)
        ctx.set_state(pos)
        p, v = ctx.get_state()
        assert not v.any()
    bad = s.pos.copy()
    bad[n // 2, 1] = np.nan
    with pytest.raises(L.NexusError) as ex:
        ctx.set_state(bad)
    assert ex.value.status == L.NX_ERR_ARG and str(3 * (n // 2) + 1) in str(ex.value)
    ctx.close()


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("passes", ["plane", "lines"])
@pytest.mark.parametrize("grid", [(8, 8, 8),        # one stage an axis
                                  (6, 15, 10),      # odd rows, lines past the last full tile
                                  (16, 27, 32),     # 4 4, 3 3 3, 4 8
                                  (128, 25, 64)])   # three stages along x, 8 8 along z
def test_transform_stages(grid, passes, prec, monkeypatch):
    monkeypatch.setenv("NEXUSMD_FFT_PLANE", "1" if passes == "plane" else "0")
    _check(_gas(411, (2.0, 2.3, 2.1), 5, grid=grid), prec, "stages %s %s" % (grid, passes))


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
def test_list_of_a_system_that_fills_the_device(prec):
    """More than 16 super-clusters per CU: the pair-list kernel's narrow blocks."""
    _check(_gas(290000, (14.2, 14.4, 14.6), 6, grid=(80, 80, 80), cutoff=0.5), prec, "full device", skin=0.05)


@pytest.mark.parametrize("prec,tol", [(L.FP64, 1e-12), (L.MIXED, 1e-6)])
@pytest.mark.parametrize("mask", [L.ALL, L.NONBONDED, L.NONBONDED | L.ANGLE, L.BOND | L.TORSION])
@pytest.mark.parametrize("n", [7, 400])
def test_terms_in_pme_launches(n, mask, prec, tol, monkeypatch):
    """Six steps with the terms in PME's launches (beside the pair kernel) and in their
    own: the same terms, so positions (nm) apart by rounding at most -- forces of
    1e4 kJ/mol/nm off by 1e-16 or 6e-8 of themselves, dt^2 / m = 4e-7."""
    s = S.bead_chain(n=n, L=2.6, grid=(24, 24, 24), seed=11)
    out = []
    for overlap in ("1", "0"):
        monkeypatch.setenv("NEXUSMD_OVERLAP", overlap)
        ctx = E.Context(s, precision=prec, skin=0.1)
        ctx.step(6, 0.0005, mask)
        out.append(np.asarray(ctx.get_state()[0]))
        ctx.close()
    print("[gpu] terms n=%d mask=%d: %.2e apart" % (n, mask, np.abs(out[0] - out[1]).max()), flush=True)
    assert np.abs(out[0] - out[1]).max() <= tol


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("grid", [(24, 24, 24), (20, 27, 25), (9, 15, 64)])
def test_planes_and_lines_give_the_same_bits(grid, prec, monkeypatch):
    """A batch takes plane or line passes by its largest system; a system's own
    numbers are the same on both."""
    s = _gas(900, (2.1, 2.3, 2.0), 3, grid=grid)
    out = []
    for passes in ("1", "0"):
        monkeypatch.setenv("NEXUSMD_FFT_PLANE", passes)
        ctx = E.Context(s, precision=prec, skin=0.1)
        ctx.step(5, 0.0005)
        out.append(np.asarray(ctx.get_state()[0]))
        ctx.close()
    np.testing.assert_array_equal(out[0], out[1])
