"""The work a user of this engine has it do, as timed cases.

Three kinds of pass, each through the Python view of the C-ABI
(`nexusmd_amd.engine`):

  md      a production loop between two reports: steps - 1 plain steps, then
          one report step that returns positions, velocities, forces and
          energies.  The trajectory continues from pass to pass.
  forces  one evaluation for an outside driver (a minimiser, a sampler, a
          rescoring script): new positions in, forces and energies out.
  serve   many small requests through the batching server: submit, run to the
          end, fetch every result.

Systems are liquids at working density with thermal velocities: flexible
water, bead chains in water (the composition of the 100,000-atom solvated
chain: one bead in ten atoms) and the bead-chain melt, tiled from one
equilibrated periodic cell per kind, moved as a whole and given fresh
velocities by the seed.  `drop` takes single water molecules out at random, so
that atom counts are odd.  Serving requests are the repository's own
ligand-in-water systems of 600 to 8,000 atoms.

The mixed path computes in 32 bits and its results are returned as float32
(trajectory frames are stored so); the FP64 path's as float64.
"""
import functools
import math

import numpy as np
import torch

from nexusmd_amd import _lib as L
from nexusmd_amd import engine as E
from nexusmd_amd import systems as S

# the cells that systems are tiled from: box edges in nm
_EDGE = {"water": 3.1, "solvated": 2.5, "chain": 4.0}

ENERGIES = ("bond", "angle", "torsion", "coulomb_direct", "lj", "recip", "self", "exclusion", "potential",
            "reference_pe", "kinetic")


def _md(name, kind, cells, precision, steps, spacing, **kw):
    c = {"name": name, "do": "md", "kind": kind, "nx": cells[0], "ny": cells[1], "nz": cells[2], "drop": 0,
         "precision": precision, "steps": steps, "spacing": spacing, "cutoff": 1.0, "skin": 0.1, "switch": 0.0}
    c.update(kw)
    return c


def listed():
    return [
        # one call of an outside driver on a small solvated system: latency and launches
        _md("forces_3k_mixed", "solvated", (2, 1, 1), "mixed", 1, 0.105, do="forces"),
        # the same on a large system in double precision, with the reference's grid rule (128^3)
        _md("forces_100k_fp64", "solvated", (4, 4, 4), "fp64", 1, 0.0, do="forces"),
        # the reference's own scale (a small protein): the 1,500-bead chain, both precisions
        _md("md_chain1500_mixed", "chain", (1, 1, 1), "mixed", 100, 0.1),
        _md("md_chain1500_fp64", "chain", (1, 1, 1), "fp64", 100, 0.1),
        # the 24,000-atom water box, 64^3: an ordinary solvated system
        _md("md_water24k_mixed", "water", (2, 2, 2), "mixed", 50, 0.0969),
        _md("md_water24k_fp64", "water", (2, 2, 2), "fp64", 50, 0.0969),
        # an oblong box with an odd atom count, a short switched cutoff and an odd grid
        _md("md_water36k_ragged", "water", (3, 2, 2), "mixed", 40, 0.125, drop=37, cutoff=0.9, skin=0.12, switch=0.75),
        # the 100,000-atom solvated chains, 96^3: the headline system
        _md("md_solvated100k_mixed", "solvated", (4, 4, 4), "mixed", 50, 0.1045),
        _md("md_solvated100k_fp64", "solvated", (4, 4, 4), "fp64", 25, 0.1045),
        # a million-atom water box, 200^3: the largest system
        _md("md_water1m_mixed", "water", (7, 7, 7), "mixed", 20, 0.1086),
        # continuous batching of small requests
        {"name": "serve_24_mixed", "do": "serve", "requests": 24, "median": 2500, "steps": 100, "precision": "mixed"},
    ]


# atoms x steps of the largest listed case, its grid counted as below
_MOST_WORK = 20 * (1_029_000 + 0.1 * 200 ** 3) * 0.8


def draw(rng):
    """One more case: every kind, size, precision and option of the listed ones."""
    do = rng.choice(("md", "md", "md", "md", "forces", "serve"))
    if do == "serve":
        return {"do": "serve", "requests": rng.randint(2, 24), "median": rng.randint(900, 3000),
                "steps": rng.randint(20, 100), "precision": "mixed"}
    kind = rng.choice(("water", "solvated", "solvated", "chain"))
    precision = rng.choice(("mixed", "mixed", "fp64"))
    weight = 3.3 if precision == "fp64" else 1.0
    atoms = math.exp(rng.uniform(math.log(1500), math.log(600_000 / weight)))
    per_cell = {"water": 3000, "solvated": 1563, "chain": 1500}[kind]
    want = max(1.0, atoms / per_cell)
    nx = max(1, round(want ** (1 / 3) * rng.uniform(0.8, 1.25)))
    ny = max(1, round((want / nx) ** 0.5 * rng.uniform(0.85, 1.2)))
    nz = max(1, round(want / (nx * ny)))
    most = int(25.6 // _EDGE[kind])            # boxes up to 25.6 nm: grids up to 256 a side
    nx, ny, nz = min(nx, most), min(ny, most), min(nz, most)
    while nx * ny * nz * per_cell * weight > 900_000:
        nz = max(1, nz - 1)
        ny = ny if nz > 1 else max(1, ny - 1)
    cutoff = rng.choice((0.9, 1.0, 1.0))
    c = {"do": do, "kind": kind, "nx": nx, "ny": ny, "nz": nz,
         "drop": rng.randint(1, 60) if kind != "chain" and rng.random() < 0.6 else 0, "precision": precision,
         "steps": 1, "spacing": rng.choice((0.0, rng.uniform(0.095, 0.125), 0.105, 0.12)), "cutoff": cutoff,
         "skin": rng.choice((0.08, 0.1, 0.1, 0.12)), "switch": cutoff - 0.15 if rng.random() < 0.25 else 0.0}
    if do == "md":
        # a grid point costs about a tenth of an atom
        cost = weight * (_atoms(c) + 0.1 * _points(c))
        c["steps"] = max(4, min(100, int(_MOST_WORK / cost), rng.randint(12, 100)))
    return c


# ------------------------------------------------------------------ systems

def _smooth(k):
    """The smallest k' >= k with prime factors 2, 3 and 5 only."""
    while True:
        m = k
        for p in (2, 3, 5):
            while m % p == 0:
                m //= p
        if m == 1:
            return k
        k += 1


def _grid(case, box):
    if case["spacing"] <= 0:
        return (0, 0, 0)           # the reference's rule, taken by the engine
    return tuple(_smooth(int(math.floor(float(b) / case["spacing"]))) for b in box)


@functools.lru_cache(maxsize=None)
def _cell(kind):
    """One equilibrated periodic cell: (box edge, positions, chain beads).

    Grown or placed on a lattice, then 500 thermostatted steps at 300 K with
    the nonbonded forces cut off and shifted inside the cell."""
    rng = np.random.default_rng({"water": 11, "solvated": 12, "chain": 13}[kind])
    edge = _EDGE[kind]
    beads = {"water": 0, "solvated": 156, "chain": 1500}[kind]
    waters = {"water": 1000, "solvated": 469, "chain": 0}[kind]
    box = np.full(3, edge)
    pos = np.zeros((0, 3))
    if beads:
        pos = S.grow_chain(beads, box, rng, min_dist=0.3) % box
    if waters:
        k = int(math.ceil(waters ** (1 / 3)))
        while True:     # the coarsest jittered lattice with room for every molecule
            a = edge / k
            g = (np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5) * a
            g += rng.uniform(-0.02, 0.02, g.shape)
            if beads:
                d = g[:, None] - pos[None]
                d -= edge * np.round(d / edge)
                g = g[(d * d).sum(-1).min(1) > 0.27 ** 2]
            if len(g) >= waters:
                break
            k += 1
        g = g[np.sort(rng.permutation(len(g))[:waters])]
        u = rng.normal(size=(waters, 2, 3))
        e1 = u[:, 0] / np.linalg.norm(u[:, 0], axis=1, keepdims=True)
        e2 = np.cross(e1, u[:, 1])
        e2 /= np.linalg.norm(e2, axis=1, keepdims=True)
        h = S.HOH_A0 / 2
        mol = np.stack([g, g + S.OH_R0 * (math.cos(h) * e1 + math.sin(h) * e2),
                        g + S.OH_R0 * (math.cos(h) * e1 - math.sin(h) * e2)], 1)
        pos = np.concatenate([pos, mol.reshape(-1, 3)])
    sys = _topology(kind, 1, pos % box, box)
    m = _Model(sys, alpha=1.5, shifted=True)
    x, v = m.tensor(sys.pos), m.tensor(S.maxwell_boltzmann(sys.mass, 300.0, rng))
    im, dt = 1.0 / m.tensor(sys.mass)[:, None], 0.0005
    for step in range(500):
        if step % 10 == 0:
            m.neighbours(x, 0.12)
        v = v + m.forces(x)[0] * im * dt
        v = v * (0.0025 / dt / (v * v).sum(1, keepdim=True).sqrt()).clamp(max=1.0)
        t = (v * v / im).sum() / (3 * sys.n * S.KB)
        v = v * (300.0 / t).sqrt().clamp(max=1.0)
        x = (x + v * dt) % m.box
    x = np.round(x.cpu().numpy(), 6)
    # whole chains and molecules, so that copies of the cell join up
    d = np.diff(x[:beads], axis=0)
    if beads:
        x[1:beads] = x[0] + np.cumsum(d - edge * np.round(d / edge), 0)
    mol = x[beads:].reshape(-1, 3, 3)
    d = mol - mol[:, :1]
    x[beads:] = (mol[:, :1] + d - edge * np.round(d / edge)).reshape(-1, 3)
    return edge, x, beads


def _topology(kind, copies, pos, box, keep=None):
    """System of `copies` cells: every chain first, then the waters (`keep`: a mask over the molecules)."""
    beads = {"water": 0, "solvated": 156, "chain": 1500}[kind]
    waters = {"water": 1000, "solvated": 469, "chain": 0}[kind]
    rng = np.random.default_rng(5)
    parts = {k: [] for k in ("b", "bp", "a", "ap", "t", "tp", "per", "q", "sig", "eps", "mass")}

    def add(**kw):
        for k, v in kw.items():
            parts[k].append(v)

    if beads:
        b, bp, a, ap, t, tp, per = S.chain_topology(beads, rng)
        q, sig, eps = S.chain_nonbonded(beads, rng)
        off = beads * np.arange(copies, dtype=np.int32)[:, None, None]
        add(b=(b[None] + off).reshape(-1, 2), bp=np.tile(bp, (copies, 1)), a=(a[None] + off).reshape(-1, 3),
            ap=np.tile(ap, (copies, 1)), t=(t[None] + off).reshape(-1, 4), tp=np.tile(tp, (copies, 1)),
            per=np.tile(per, copies), q=np.tile(q, copies), sig=np.tile(sig, copies), eps=np.tile(eps, copies),
            mass=np.full(beads * copies, S.BEAD_MASS))
    n_mol = waters * copies if keep is None else int(keep.sum())
    if n_mol:
        b, bp, a, ap, q, sig, eps, mass = S.water_topology(n_mol, beads * copies, h_core=beads > 0)
        add(b=b, bp=bp, a=a, ap=ap, q=q, sig=sig, eps=eps, mass=mass)
    c = {k: np.concatenate(v) if v else None for k, v in parts.items()}
    none = np.zeros(0, np.int32)
    return S.System("%s_%d" % (kind, len(pos)), pos, np.zeros_like(pos), c["mass"], c["b"], c["bp"], c["a"], c["ap"],
                    c["t"] if c["t"] is not None else none.reshape(0, 4),
                    c["tp"] if c["tp"] is not None else np.zeros((0, 2)),
                    c["per"] if c["per"] is not None else none, c["q"], c["sig"], c["eps"], np.zeros(3),
                    np.array(box, float))


def _system(case, seed):
    edge, cell, beads = _cell(case["kind"])
    rng = np.random.default_rng(seed)
    shape = (case["nx"], case["ny"], case["nz"])
    box = edge * np.array(shape, float)
    at = np.stack(np.meshgrid(*[np.arange(s) for s in shape], indexing="ij"), -1).reshape(-1, 1, 3) * edge
    copies = len(at)
    chains = (cell[None, :beads] + at).reshape(-1, 3)
    mols = (cell[None, beads:] + at).reshape(-1, 3, 3)
    keep = np.ones(len(mols), bool)
    keep[rng.permutation(len(mols))[:case["drop"]]] = False
    pos = np.concatenate([chains, mols[keep].reshape(-1, 3)])
    # the seed's own liquid: moved as a whole, thermal noise, velocities
    pos = (pos + rng.uniform(0, 1, 3) * box + rng.normal(0.0, 0.0005, pos.shape)) % box
    sys = _topology(case["kind"], copies, pos, box, keep)
    sys.vel = S.maxwell_boltzmann(sys.mass, 300.0, rng)
    sys.cutoff = case["cutoff"]
    sys.grid = _grid(case, box)
    sys.dt = 0.0005
    return sys


@functools.lru_cache(maxsize=64)
def _ligands(requests, median):
    """Ligand-in-water systems, lognormal sizes within the serving range."""
    rng = np.random.default_rng(requests * 10_000 + median)
    sizes = np.clip(np.exp(rng.normal(math.log(median), 0.6, requests)), 600, 8000).astype(int)
    return [S.ligand_in_water(int(n), int(rng.integers(1 << 31))) for n in sizes]


def _requests(case, seed):
    """The case's requests, each moved as a whole and with velocities of its own."""
    rng, out = np.random.default_rng(seed), []
    for s in _ligands(case["requests"], case["median"]):
        s = s.copy()
        s.pos = (s.pos + rng.uniform(0, 1, 3) * s.L + rng.normal(0.0, 0.0005, s.pos.shape)) % s.L
        s.vel = S.maxwell_boltzmann(s.mass, 300.0, rng)
        out.append(s)
    return out


# -------------------------------------------------------------------- passes

def _precision(case):
    return L.MIXED if case["precision"] == "mixed" else L.FP64


def prepare(case, seed):
    real = np.float32 if case["precision"] == "mixed" else np.float64
    if case["do"] == "serve":
        return {"do": "serve", "real": real, "systems": _requests(case, seed), "steps": case["steps"],
                "server": E.Server(precision=_precision(case), max_active=case["requests"])}
    sys = _system(case, seed)
    ctx = E.Context(sys, precision=_precision(case), skin=case["skin"], use_switch=int(case["switch"] > 0),
                    switch_distance=case["switch"])
    return {"do": case["do"], "real": real, "ctx": ctx, "pos": sys.pos, "steps": case["steps"], "dt": sys.dt}


def _energies(e, real):
    return np.array([e[k] for k in ENERGIES], real)


def run(state):
    real = state["real"]
    if state["do"] == "serve":
        server = state["server"]
        ids = [server.submit(s, state["steps"], s.dt) for s in state["systems"]]
        server.run()
        got = [server.fetch(i) for i in ids]
        return {"positions": np.concatenate([p for p, _, _ in got]).astype(real),
                "velocities": np.concatenate([v for _, v, _ in got]).astype(real),
                "energies": np.stack([_energies(e, real) for _, _, e in got])}
    ctx = state["ctx"]
    if state["do"] == "forces":
        ctx.set_state(state["pos"])
        f, e = ctx.compute_forces()
        return {"forces": f.astype(real), "energies": _energies(e, real)}
    ctx.step(state["steps"] - 1, state["dt"])
    p, v, f, e = ctx.step_report(state["dt"])
    return {"positions": p.astype(real), "velocities": v.astype(real), "forces": f.astype(real),
            "energies": _energies(e, real)}


def _atoms(case):
    per = {"water": 3000, "solvated": 1563, "chain": 1500}[case["kind"]]
    return per * case["nx"] * case["ny"] * case["nz"] - 3 * case["drop"]


def _points(case):
    """Points of the PME grid."""
    box = [_EDGE[case["kind"]] * case[k] for k in ("nx", "ny", "nz")]
    g = _grid(case, box)
    if g[0] == 0:
        g = [1 << (10 * math.ceil(b) - 1).bit_length() for b in box]
    return float(g[0] * g[1] * g[2])


def work(case):
    """Per step: the state read and written in 64 bits, 75 FLOP a pair inside
    the cutoff, the order-5 spread and gather, two real 3D FFTs."""
    if case["do"] == "serve":
        n = case["requests"] * case["median"] * 1.2      # the mean of the lognormal sizes
        rho, grid, steps, cutoff = 100.0, n * 8.0, case["steps"], 0.9
    else:
        n, steps, cutoff = _atoms(case), case["steps"], case["cutoff"]
        rho = n / (_EDGE[case["kind"]] ** 3 * case["nx"] * case["ny"] * case["nz"])
        grid = _points(case)
    pairs = 0.5 * n * rho * 4.0 / 3.0 * math.pi * cutoff ** 3
    flops = steps * (75.0 * pairs + n * 125 * 8.0 + 2 * 2.5 * grid * math.log2(max(2.0, grid)))
    bytes_ = steps * n * 96.0
    return {"bytes": bytes_, "flops": flops}


# ---------------------------------------------------- the same in 64 bits
#
# Plain torch on the GPU (the CPU without one): harmonic bonds and angles,
# periodic torsions, Lennard-Jones and Ewald direct space inside the cutoff
# from a padded neighbour table, the exclusion correction, order-5 smooth PME
# through torch.fft, leapfrog.

_KE = 138.93545764446428693393


def _rows(index, n_rows, n_cols_min=1):
    """Padded table: row r holds the positions k with index[k] == r (ascending), -1 elsewhere."""
    order = torch.argsort(index, stable=True)
    counts = torch.bincount(index, minlength=n_rows)
    first = torch.cumsum(counts, 0) - counts
    col = torch.arange(len(index), device=index.device) - first[index[order]]
    table = torch.full((n_rows, max(n_cols_min, int(counts.max()) if len(index) else 1)), -1, dtype=torch.int64,
                       device=index.device)
    table[index[order], col] = order
    return table


class _Model:
    def __init__(self, sys, alpha=None, shifted=False):
        self.device = "cuda" if torch.cuda.is_available() else "cpu"
        t = self.tensor
        self.sys, self.n, self.box = sys, sys.n, t(sys.L)
        self.rc = float(sys.cutoff)
        self.alpha = alpha or math.sqrt(-math.log(2 * sys.ewald_tol)) / self.rc
        self.shifted, self.switch = shifted, 0.0
        self.q, self.sig, self.e2 = t(sys.q), t(sys.sig) / 2, 2 * t(sys.eps).sqrt()
        self.mass = t(sys.mass)
        idx = lambda a, k: torch.as_tensor(np.asarray(a, np.int64).reshape(-1, k), device=self.device)  # noqa: E731
        self.b, self.bp = idx(sys.bond_idx, 2), t(sys.bond_par).reshape(-1, 2)
        self.a, self.ap = idx(sys.angle_idx, 3), t(sys.angle_par).reshape(-1, 2)
        self.t, self.tp = idx(sys.torsion_idx, 4), t(sys.torsion_par).reshape(-1, 2)
        self.per = t(sys.torsion_per)
        # which term-force rows act on each atom
        self.term_of = _rows(torch.cat([self.b.reshape(-1), self.a.reshape(-1), self.t.reshape(-1)]), self.n)
        # pairs up to three bonds apart, as sorted keys i n + j (both orders)
        up = torch.cat([self.b, self.b.flip(1)])
        near = _rows(up[:, 0], self.n)
        near = torch.where(near >= 0, up[near.clamp(min=0), 1], torch.full_like(near, -1))
        me = torch.arange(self.n, device=self.device)[:, None]
        ring, keys = near, []
        for depth in range(3):
            pair = me.expand_as(ring)[(ring >= 0) & (ring != me)] * self.n + ring[(ring >= 0) & (ring != me)]
            keys.append(pair)
            if depth < 2:
                ring = torch.where((ring >= 0)[:, :, None], near[ring.clamp(min=0)], torch.full_like(near[:1, None, :1], -1))
                ring = ring.reshape(self.n, -1)
        self.excl = torch.unique(torch.cat(keys))

    def tensor(self, a):
        return torch.as_tensor(np.asarray(a, np.float64), device=self.device)

    def image(self, d):
        return d - self.box * torch.round(d / self.box)

    def _excluded(self, i, j):
        if not len(self.excl):
            return torch.zeros_like(i, dtype=torch.bool)
        key = i * self.n + j
        at = torch.searchsorted(self.excl, key).clamp(max=len(self.excl) - 1)
        return self.excl[at] == key

    def neighbours(self, x, margin):
        """self.nb: padded table of the partners within the cutoff plus `margin`, exclusions left out."""
        r2 = (self.rc + margin) ** 2
        cells = [int(b // math.sqrt(r2)) for b in self.box.tolist()]
        found_i, found_j = [], []

        def keep(i, j):
            sel = ~self._excluded(i, j)
            found_i.append(i[sel].to(torch.int32))
            found_j.append(j[sel].to(torch.int32))

        if min(cells) < 3 or self.n < 20000:
            rows = max(1, int(1.5e8 // (3 * self.n)))
            for at in range(0, self.n, rows):
                d = self.image(x[at:at + rows, None] - x[None])
                i, j = torch.nonzero((d * d).sum(-1) < r2, as_tuple=True)
                i = i + at
                keep(i[i != j], j[i != j])
        else:
            nc = torch.tensor(cells, device=self.device)
            c = torch.minimum((x / self.box * nc).long().clamp(min=0), nc - 1)
            flat = (c[:, 0] * cells[1] + c[:, 1]) * cells[2] + c[:, 2]
            table = _rows(flat, cells[0] * cells[1] * cells[2])
            pad = torch.cat([x, torch.full((1, 3), 1e6, device=self.device, dtype=x.dtype)])
            cap = table.shape[1]
            rows = max(1, int(6e7 // (cap * cap)))
            steps = [torch.tensor((a, b, g), device=self.device) for a in (-1, 0, 1) for b in (-1, 0, 1) for g in (-1, 0, 1)]
            for at in range(0, table.shape[0], rows):
                own = torch.arange(at, min(at + rows, table.shape[0]), device=self.device)
                c3 = torch.stack([own // (cells[1] * cells[2]), own // cells[2] % cells[1], own % cells[2]], 1)
                mine = table[own]
                for s in steps:
                    o = (c3 + s) % nc
                    other = table[(o[:, 0] * cells[1] + o[:, 1]) * cells[2] + o[:, 2]]
                    d = pad[mine][:, :, None] - pad[other][:, None]
                    d = self.image(d)
                    ok = ((d * d).sum(-1) < r2) & (mine >= 0)[:, :, None] & (other >= 0)[:, None]
                    k, u, w = torch.nonzero(ok, as_tuple=True)
                    i, j = mine[k, u], other[k, w]
                    keep(i[i != j], j[i != j])
        i, j = torch.cat(found_i).long(), torch.cat(found_j)
        table = _rows(i, self.n)
        self.nb = torch.where(table >= 0, j[table.clamp(min=0)].long(), torch.full_like(table, -1)) if len(i) else table
        self.nb_at = x.clone()

    def direct(self, x):
        f, ec, el = torch.zeros_like(x), x.new_zeros(()), x.new_zeros(())
        a, rc = self.alpha, self.rc
        rows = max(1, int(2e7 // self.nb.shape[1]))
        if self.shifted:
            f_rc = math.erfc(a * rc) / rc ** 2 + 2 * a / math.sqrt(math.pi) * math.exp(-(a * rc) ** 2) / rc
        for at in range(0, self.n, rows):
            j = self.nb[at:at + rows]
            on = j >= 0
            j = j.clamp(min=0)
            d = self.image(x[at:at + rows, None] - x[j])
            r2 = (d * d).sum(-1)
            on = on & (r2 < rc * rc)
            r2 = torch.where(on, r2, torch.ones_like(r2))
            r = r2.sqrt()
            qq = _KE * self.q[at:at + rows, None] * self.q[j]
            s6 = ((self.sig[at:at + rows, None] + self.sig[j]) ** 2 / r2) ** 3
            ep = self.e2[at:at + rows, None] * self.e2[j]
            erfc = torch.erfc(a * r)
            coul = qq * erfc / r
            fc = qq / r * (erfc / r2 + 2 * a / math.sqrt(math.pi) * torch.exp(-a * a * r2) / r)
            if self.shifted:
                fc = fc - qq * f_rc / r
            lj = ep * (s6 - 1) * s6
            fl = ep * (12 * s6 - 6) * s6 / r2
            if self.switch > 0:
                t = ((r - self.switch) / (rc - self.switch)).clamp(min=0.0)
                sv = 1 + t ** 3 * (-10 + t * (15 - 6 * t))
                sd = t * t * (-30 + t * (60 - 30 * t)) / (rc - self.switch)
                fl = sv * fl - lj * sd / r
                lj = lj * sv
            g = torch.where(on, fc + fl, torch.zeros_like(fc))
            f[at:at + rows] = (d * g[:, :, None]).sum(1)
            ec = ec + 0.5 * torch.where(on, coul, torch.zeros_like(coul)).sum()
            el = el + 0.5 * torch.where(on, lj, torch.zeros_like(lj)).sum()
        return f, ec, el

    def terms(self, x):
        """Bonds, angles, torsions: forces and the three energies."""
        rows, e = [], [x.new_zeros(())] * 3
        if len(self.b):
            d = self.image(x[self.b[:, 1]] - x[self.b[:, 0]])
            r = d.norm(dim=1)
            off = r - self.bp[:, 0]
            f = d * (self.bp[:, 1] * off / r)[:, None]
            rows.append(torch.stack([f, -f], 1).reshape(-1, 3))
            e[0] = (0.5 * self.bp[:, 1] * off * off).sum()
        if len(self.a):
            u = self.image(x[self.a[:, 1]] - x[self.a[:, 0]])
            w = self.image(x[self.a[:, 1]] - x[self.a[:, 2]])
            c = torch.linalg.cross(u, w)
            rp = c.norm(dim=1).clamp(min=1e-6)
            off = torch.atan2(rp, (u * w).sum(1)) - self.ap[:, 0]
            g = self.ap[:, 1] * off
            f1 = torch.linalg.cross(u, c) * (g / ((u * u).sum(1) * rp))[:, None]
            f3 = torch.linalg.cross(c, w) * (g / ((w * w).sum(1) * rp))[:, None]
            rows.append(torch.stack([f1, -f1 - f3, f3], 1).reshape(-1, 3))
            e[1] = (0.5 * self.ap[:, 1] * off * off).sum()
        if len(self.t):
            u = self.image(x[self.t[:, 0]] - x[self.t[:, 1]])
            w = self.image(x[self.t[:, 2]] - x[self.t[:, 1]])
            z = self.image(x[self.t[:, 2]] - x[self.t[:, 3]])
            c0, c1 = torch.linalg.cross(u, w), torch.linalg.cross(w, z)
            lw = w.norm(dim=1)
            phi = torch.atan2(lw * (u * c1).sum(1), (c0 * c1).sum(1))
            arg = self.per * phi - self.tp[:, 1]
            g = -self.tp[:, 0] * self.per * torch.sin(arg)
            f1 = c0 * (-g * lw / (c0 * c0).sum(1))[:, None]
            f4 = c1 * (g * lw / (c1 * c1).sum(1))[:, None]
            s = f1 * ((u * w).sum(1) / lw ** 2)[:, None] - f4 * ((z * w).sum(1) / lw ** 2)[:, None]
            rows.append(torch.stack([f1, s - f1, -s - f4, f4], 1).reshape(-1, 3))
            e[2] = (self.tp[:, 0] * (1 + torch.cos(arg))).sum()
        if not rows:
            return torch.zeros_like(x), e
        rows = torch.cat(rows + [x.new_zeros((1, 3))])
        return rows[self.term_of].sum(1), e        # -1: the zero row

    def forces(self, x):
        """Without PME: what equilibrates a cell."""
        f, ec, el = self.direct(x)
        g, e = self.terms(x)
        return f + g, ec, el, e

    # ------------------------------------------------------- with PME

    def set_pme(self, grid):
        n = [int(k) for k in grid]
        if n[0] == 0:
            n = [1 << (10 * math.ceil(b) - 1).bit_length() for b in self.box.tolist()]
        self.grid = n
        box, mod, m = self.box.tolist(), [], []
        for k in n:
            w = np.zeros(max(k, 6))
            w[1:5] = np.array([1.0, 11.0, 11.0, 1.0]) / 24.0       # the order-5 spline at the integers
            b = np.abs(np.fft.fft(w)) ** 2 if len(w) == k else np.abs(
                np.exp(-2j * np.pi * np.outer(np.arange(k), np.arange(k)) / k) @ w[:k]) ** 2
            for i in range(k):
                if b[i] < 1e-7:
                    b[i] = 0.5 * (b[i - 1] + b[(i + 1) % k])
            mod.append(self.tensor(b))
            m.append(self.tensor(np.where(np.arange(k) < (k + 1) // 2, np.arange(k), np.arange(k) - k)))
        h = n[2] // 2 + 1
        m2 = ((m[0] / box[0])[:, None, None] ** 2 + (m[1] / box[1])[None, :, None] ** 2 +
              (m[2][:h] / box[2])[None, None] ** 2)
        m2[0, 0, 0] = 1.0
        vol = box[0] * box[1] * box[2]
        eta = _KE * torch.exp(-(math.pi / self.alpha) ** 2 * m2) / (
            m2 * math.pi * vol * mod[0][:, None, None] * mod[1][None, :, None] * mod[2][None, None, :h])
        eta[0, 0, 0] = 0.0
        self.eta = eta
        self.ew = torch.full((h,), 1.0, dtype=torch.float64, device=self.device)
        self.ew[0] = 0.5
        if n[2] % 2 == 0:
            self.ew[-1] = 0.5
        self.ei, self.ej = self.excl // self.n, self.excl % self.n
        self.excl_of = _rows(self.ei, self.n) if len(self.excl) else None

    @staticmethod
    def _spline(f):
        """Order-5 B-spline weights and derivatives at fraction f: [..., 5] each."""
        t = [1 - f, f]
        for k in range(3, 6):
            if k == 5:
                low = t
            t = [((1 - f) * t[0]) / (k - 1)] + [
                ((f + k - 1 - i) * t[i - 1] + (i + 1 - f) * t[i]) / (k - 1) for i in range(1, k - 1)
            ] + [f * t[-1] / (k - 1)]
        d = [-low[0]] + [low[i - 1] - low[i] for i in range(1, 4)] + [low[3]]
        return torch.stack(t, -1), torch.stack(d, -1)

    def recip(self, x):
        n = self.grid
        k = torch.tensor(n, device=self.device)
        s = x / self.box
        s = (s - torch.floor(s)) * k
        base = s.long()
        th, dth = self._spline(s - base)
        o = torch.arange(5, device=self.device)
        i = [(base[:, c, None] + o) % n[c] for c in range(3)]
        grid = torch.zeros(n[0] * n[1] * n[2], dtype=torch.float64, device=self.device)
        rows = 200000
        for at in range(0, self.n, rows):
            u = slice(at, at + rows)
            cell = ((i[0][u, :, None, None] * n[1] + i[1][u, None, :, None]) * n[2] + i[2][u, None, None]).reshape(-1)
            w = (self.q[u, None, None, None] * th[u, 0, :, None, None] * th[u, 1, None, :, None] *
                 th[u, 2, None, None, :]).reshape(-1)
            grid.index_add_(0, cell, w)
        c = torch.fft.rfftn(grid.reshape(n))
        e = (self.eta * self.ew * (c.real ** 2 + c.imag ** 2)).sum()
        phi = (torch.fft.irfftn(c * self.eta, s=n) * float(n[0] * n[1] * n[2])).reshape(-1)
        f = torch.empty_like(x)
        for at in range(0, self.n, rows):
            u = slice(at, at + rows)
            v = phi[(i[0][u, :, None, None] * n[1] + i[1][u, None, :, None]) * n[2] + i[2][u, None, None]]
            w = [(dth if c == a else th)[u, c] for a in range(3) for c in range(3)]
            for a in range(3):
                x3, y3, z3 = w[3 * a:3 * a + 3]
                g = (v * x3[:, :, None, None] * y3[:, None, :, None] * z3[:, None, None, :]).sum((1, 2, 3))
                f[u, a] = -self.q[u] * g * (n[a] / float(self.box[a]))
        return f, e

    def full(self, x):
        """Forces and the energies of ENERGIES (without the kinetic one)."""
        if getattr(self, "nb", None) is None or float((self.image(x - self.nb_at) ** 2).sum(1).max()) > 0.07 ** 2:
            self.neighbours(x, 0.15)
        f, ec, el = self.direct(x)
        g, e = self.terms(x)
        h, er = self.recip(x)
        f = f + g + h
        a = self.alpha
        es = -_KE * a / math.sqrt(math.pi) * (self.q ** 2).sum()
        ex = x.new_zeros(())
        if self.excl_of is not None:
            d = self.image(x[self.ei] - x[self.ej])
            r = d.norm(dim=1)
            qq = _KE * self.q[self.ei] * self.q[self.ej]
            ef = torch.erf(a * r)
            w = qq / r ** 3 * (ef - 2 * a * r * torch.exp(-(a * r) ** 2) / math.sqrt(math.pi))
            row = torch.cat([-d * w[:, None], x.new_zeros((1, 3))])
            f = f + row[self.excl_of].sum(1)
            ex = 0.5 * (qq * ef / r).sum()
        bonded = e[0] + e[1] + e[2]
        nonbonded = er + es + ec + el - ex
        return f, [e[0], e[1], e[2], ec, el, er, es, ex, bonded + nonbonded, nonbonded]

    def advance(self, x, v, f, dt):
        v = v + f / self.mass[:, None] * dt
        x = x + v * dt
        x = torch.where(x < 0, x + self.box, torch.where(x > self.box, x - self.box, x))
        return x, v


def _numbers(e, kinetic):
    return np.array([float(t) for t in e] + [float(kinetic)])


def exact(case, seed):
    if case["do"] == "serve":
        if case["requests"] * case["steps"] > 2500:
            return None
        p, v, e = [], [], []
        for s in _requests(case, seed):
            m = _Model(s)
            m.set_pme(s.grid)
            x, u = m.tensor(s.pos), m.tensor(s.vel)
            for _ in range(case["steps"]):
                x, u = m.advance(x, u, m.full(x)[0], s.dt)
            p.append(x.cpu().numpy())
            v.append(u.cpu().numpy())
            e.append(_numbers(m.full(x)[1], 0.0))
        return {"positions": np.concatenate(p), "velocities": np.concatenate(v), "energies": np.stack(e)}
    s = _system(case, seed)
    m = _Model(s)
    m.switch = case["switch"]
    m.set_pme(s.grid)
    x, v = m.tensor(s.pos), m.tensor(s.vel)
    if case["do"] == "forces":
        f, e = m.full(x)
        return {"forces": f.cpu().numpy(), "energies": _numbers(e, 0.0)}
    for _ in range(case["steps"] - 1):
        x, v = m.advance(x, v, m.full(x)[0], s.dt)
    f, e = m.full(x)
    half = v + f / m.mass[:, None] * (0.5 * s.dt)
    kinetic = 0.5 * (m.mass[:, None] * half * half).sum()
    return {"positions": x.cpu().numpy(), "velocities": v.cpu().numpy(), "forces": f.cpu().numpy(),
            "energies": _numbers(e, kinetic)}
