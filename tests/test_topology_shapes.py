"""Topology arrays that are too short, too narrow or wider than their records (CPU)."""
import numpy as np
import pytest

from nexusmd_amd import engine as E
from nexusmd_amd import systems as S


def _chain():
    return S.bead_chain(40, 2.2, seed=3)


@pytest.mark.parametrize("name", ["bond_par", "angle_par", "torsion_par", "torsion_per"])
def test_one_row_of_parameters_does_not_stand_for_all(name):
    s = _chain()
    setattr(s, name, getattr(s, name)[:1])
    with pytest.raises(IndexError):
        E.TopologyBuffers(s)


@pytest.mark.parametrize("name", ["bond_par", "angle_par", "torsion_par"])
def test_a_missing_parameter_column_raises(name):
    s = _chain()
    setattr(s, name, getattr(s, name)[:, :1])
    with pytest.raises(IndexError):
        E.TopologyBuffers(s)


@pytest.mark.parametrize("name", ["bond_idx", "angle_idx", "torsion_idx"])
@pytest.mark.parametrize("change", ["one less", "one more"])
def test_another_number_of_particles_raises(name, change):
    s = _chain()
    a = getattr(s, name)
    setattr(s, name, a[:, :-1] if change == "one less" else np.hstack([a, a[:, :1]]))
    with pytest.raises(ValueError):
        E.TopologyBuffers(s)


def test_what_follows_the_records_is_not_read():
    """Rows past the last record and columns past the last field, whole numbers given
    as floats: the same records."""
    s, t = _chain(), _chain()
    for name in ("bond_par", "angle_par", "torsion_par"):
        a = getattr(t, name)
        setattr(t, name, np.vstack([np.hstack([a, np.full((len(a), 1), np.nan)]), np.full((2, a.shape[1] + 1), np.nan)]))
    t.torsion_per = np.concatenate([t.torsion_per.astype(float), [np.nan]])
    t.bond_idx = t.bond_idx.astype(float)
    a, b = E.TopologyBuffers(s), E.TopologyBuffers(t)
    for x, y in ((a.bonds, b.bonds), (a.angles, b.angles), (a.torsions, b.torsions)):
        assert bytes(x) == bytes(y)


def test_an_index_that_is_not_a_number_raises():
    s = _chain()
    s.bond_idx = s.bond_idx.astype(float)
    s.bond_idx[3, 1] = np.nan
    with pytest.raises(ValueError):
        E.TopologyBuffers(s)
