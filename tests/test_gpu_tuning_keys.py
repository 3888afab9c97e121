"""Keys under which tuned launch shapes are kept."""
import pytest

from nexusmd_amd import _lib as L
from nexusmd_amd import engine as E
from nexusmd_amd import systems as S

pytestmark = pytest.mark.gpu


def test_tuned_shapes_of_one_pair_kernel_are_not_taken_for_the_other(tmp_path, monkeypatch):
    """Two FP64 systems that differ in the Ewald tolerance alone, either side of the
    range where the pair kernel needs library functions: two keys in the cache."""
    path = tmp_path / "tuned"
    monkeypatch.setenv("NEXUSMD_TUNE_CACHE", str(path))
    for tol in (1.7e-4, 1.6e-4):
        s = S.water_box(n_mol=300, L=2.1, grid=(20, 20, 24), seed=14)
        s.ewald_tol = tol
        print("[gpu] autotune at tolerance %g" % tol, flush=True)
        ctx = E.Context(s, precision=L.FP64, skin=0.1)
        ctx.autotune(steps_per_trial=4)
        ctx.close()
    keys = [line.split("\t")[0] for line in path.read_text().splitlines()]
    assert len(keys) == 2 and keys[0] != keys[1]
