"""FP64 forces either side of the sizes where the pair kernel takes longer chunks,
against the FP64 oracle (relative RMS 1e-9, the bound of the other parity tests)."""
import numpy as np
import pytest

from nexusmd_amd import _lib as L
from nexusmd_amd import engine as E
from oracle import pyoracle as O

from _util import bare_system, rel_rms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16499, 16500, 41999, 42000])
def test_fp64_chunk_lengths(n):
    rng = np.random.default_rng(n)
    box = np.array([5.0, 5.5, 6.0]) * (n / 16500) ** (1 / 3)
    k = np.ceil(box * (n / box.prod()) ** (1 / 3)).astype(int)
    while k.prod() < n:
        k[np.argmin(k / box)] += 1
    g = np.stack(np.meshgrid(*[np.arange(m) + 0.5 for m in k], indexing="ij"), -1).reshape(-1, 3) * (box / k)
    pos = (g[rng.permutation(len(g))[:n]] + rng.normal(0.0, 0.01, (n, 3))) % box
    q = rng.normal(0.0, 0.4, n)
    s = bare_system(pos, np.zeros(3), box, q=q - q.mean(), sig=np.full(n, 0.12), eps=rng.uniform(0.1, 0.4, n),
                    cutoff=0.7, grid=(40, 40, 48))
    print("[gpu] chunk lengths n=%d" % n, flush=True)
    ctx = E.Context(s, precision=L.FP64, skin=0.1)
    f, _ = ctx.compute_forces()
    ctx.close()
    ref, _ = O.compute_forces(O.Prepared(s))
    assert rel_rms(f, ref) <= 1e-9
