"""Records of the topology and the exclusion lists against straightforward loops (CPU)."""
import numpy as np
import pytest

from nexusmd_amd import _lib as L
from nexusmd_amd import engine as E
from nexusmd_amd import systems as S


@pytest.mark.parametrize("sys", [S.bead_chain(40, 2.2, seed=3), S.water_box(30, 1.2, seed=4)], ids=["chain", "water"])
def test_topology_records(sys):
    b = E.TopologyBuffers(sys)
    for t in range(len(sys.bond_idx)):
        assert (b.bonds[t].p1, b.bonds[t].p2, b.bonds[t].d, b.bonds[t].k) == (*sys.bond_idx[t], *sys.bond_par[t])
    for t in range(len(sys.angle_idx)):
        assert (b.angles[t].p1, b.angles[t].p2, b.angles[t].p3, b.angles[t].a, b.angles[t].k) == \
            (*sys.angle_idx[t], *sys.angle_par[t])
    for t in range(len(sys.torsion_idx)):
        x = b.torsions[t]
        assert (x.p1, x.p2, x.p3, x.p4, x.k, x.phase, x.periodicity) == \
            (*sys.torsion_idx[t], *sys.torsion_par[t], sys.torsion_per[t])
    assert (len(b.bonds), len(b.angles), len(b.torsions)) == tuple(
        max(1, len(a)) for a in (sys.bond_idx, sys.angle_idx, sys.torsion_idx))
    assert isinstance(b.bonds[0], L.Bond)
