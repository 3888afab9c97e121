"""Systems at the room that a layout leaves them: crowded columns, lists that grow
after the layout, exclusions by the hundred in one super-cluster.

Forces against the FP64 oracle, relative RMS: FP64 <= 1e-9, mixed <= 5e-4 (the
bounds of the other parity tests).
"""
import numpy as np
import pytest

from nexusmd_amd import _lib as L
from nexusmd_amd import engine as E
from oracle import pyoracle as O

from _util import bare_system, rel_rms

pytestmark = pytest.mark.gpu

TOL = {L.FP64: 1e-9, L.MIXED: 5e-4}


def _lattice(n, box, rng):
    """n jittered lattice points in [0, box)."""
    box = np.asarray(box, float)
    k = np.ceil(box * (n / box.prod()) ** (1 / 3)).astype(int)
    while k.prod() < n:
        k[np.argmin(k / box)] += 1
    g = np.stack(np.meshgrid(*[np.arange(m) + 0.5 for m in k], indexing="ij"), -1).reshape(-1, 3) * (box / k)
    return g[rng.permutation(len(g))[:n]] + rng.normal(0.0, 0.01, (n, 3))


def _gas(n, box, rng, grid, cutoff=0.8):
    q = rng.normal(0.0, 0.4, n)
    return bare_system(_lattice(n, box, rng) % box, np.zeros(3), box, q=q - q.mean(), sig=np.full(n, 0.12),
                       eps=rng.uniform(0.1, 0.4, n), cutoff=cutoff, grid=grid)


def _same(sys, prec, f, pos, excl=None):
    sys.pos = pos
    ref, _ = O.compute_forces(O.Prepared(sys, excl=excl))
    assert rel_rms(f, ref) <= TOL[prec]


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("layout", ["spread out", "clumped"])
def test_a_clump_across_columns(layout, prec):
    """2,100 of 2,800 atoms in one quarter of the xy plane, under 1,000 in every cell
    of the 3 x 3 that a column of 8-atom clusters would have here: as the first
    state, and as a later state of a context laid out for an even one."""
    rng = np.random.default_rng(1)
    box = np.array([1.95, 1.95, 11.5])
    s = _gas(2800, box, rng, (24, 24, 128))
    even = s.pos.copy()
    dense = np.vstack([_lattice(2100, box * [0.5, 0.5, 1.0], rng), _lattice(700, box * [0.5, 1.0, 1.0], rng) + box * [0.5, 0, 0]])
    dense %= box
    cell = (dense[:, :2] / box[:2] * 3).astype(int)
    assert np.bincount(cell[:, 0] * 3 + cell[:, 1]).max() < 2048
    print("[gpu] clump, first %s, precision %d" % (layout, prec), flush=True)
    if layout == "clumped":
        s.pos = dense
    ctx = E.Context(s, precision=prec, skin=0.1)
    ctx.compute_forces()
    ctx.set_state(dense)
    f, _ = ctx.compute_forces()
    ctx.close()
    s.pos = even
    _same(s, prec, f, dense)


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
def test_a_gas_that_condenses(prec):
    """4,000 atoms at 1 in 2 nm^3, then as a drop of 60 per nm^3 in the same context:
    the pair list has room for it."""
    rng = np.random.default_rng(2)
    box = np.array([20.0, 20.0, 20.0])
    s = _gas(4000, box, rng, (64, 64, 64), cutoff=1.0)
    print("[gpu] condensing gas, precision %d" % prec, flush=True)
    ctx = E.Context(s, precision=prec, skin=0.1)
    ctx.compute_forces()
    drop = _lattice(4000, (4.05, 4.05, 4.05), rng) + 7.9
    ctx.set_state(drop)
    f, _ = ctx.compute_forces()
    ctx.close()
    _same(s, prec, f, drop)


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("group", [60, 80])
def test_a_group_without_interactions_inside(group, prec):
    """`group` neighbouring atoms around the middle of a column, every pair of them
    excluded, in a box of 900: with 80, some 2,700 excluded pairs in one
    super-cluster."""
    rng = np.random.default_rng(3)
    box = np.array([2.4, 2.3, 2.2])
    s = _gas(900, box, rng, (24, 24, 24))
    d = s.pos - box * [0.25, 0.25, 0.5]
    order = np.argsort((d * d).sum(1))
    s.pos = s.pos[order]
    s.q = s.q[order]
    s.eps = s.eps[order]
    off = np.concatenate([np.arange(group + 1) * (group - 1), np.full(900 - group, group * (group - 1))]).astype(np.int32)
    idx = np.concatenate([[j for j in range(group) if j != i] for i in range(group)]).astype(np.int32)
    print("[gpu] %d atoms excluded from each other, precision %d" % (group, prec), flush=True)
    ctx = E.Context(s, precision=prec, skin=0.1, excl=(off, idx))
    f, _ = ctx.compute_forces()
    pairs = ctx.neighbor_pairs() if prec == L.FP64 else None
    ctx.close()
    _same(s, prec, f, s.pos, excl=(off, idx))
    if pairs is not None:
        want = O.pairs(s, (off, idx), method="brute")
        assert set(map(tuple, pairs.tolist())) == set(map(tuple, want.tolist()))
