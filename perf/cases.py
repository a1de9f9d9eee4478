"""The work that programs have this framework do, as measurable cases.

Four kinds of call, all through ``dftbplus_amd.api``:

* ``point``: one geometry step of a resident calculator - new coordinates, a fixed number of SCC
  iterations, energy, charges, levels and forces (a molecular-dynamics or relaxation step).
  Clusters, periodic cells at the Gamma point, k-point meshes; FP64 and mixed precision.
* ``tail``: the same step in mixed precision, started from the charges of the geometry step
  before, so that its iterations refine eigenvectors instead of solving for them.
* ``batch``: many independent molecules set up, iterated and differentiated together.
* ``dense``: the drop-ins that a host program calls in place of its own eigensolver and density
  matrix routines (real or complex, host arrays in and out).

Geometries and Slater-Koster sets are the synthetic recipes of ``dftbplus_amd.synth``. The SCC
iteration count of a pass is fixed, so a pass does the same work whatever the last bits are.
``exact`` restates the calculation in float64 (dense pair lists, Lagrange interpolation, gradients
by differentiating the energy functional at fixed density), without the framework's code.
"""
import dataclasses
import math

import numpy as np
import torch

from dftbplus_amd import api, synth
from dftbplus_amd.model import Geometry, Options

# Broyden parameter and electron temperature of each recipe: those of the workloads of the same
# recipes; the cluster is run at about 300 K.
RECIPES = {"cluster": (1.0e-3, 0.2, 100), "diamond": (1.0e-2, 0.05, 101),
           "water": (3.0e-3, 0.05, 102), "amorphous": (1.0e-3, 0.2, 104)}
ELEMENTS = {"cluster": ["H", "C", "O"], "diamond": ["C", "H", "O"], "water": ["O", "H"],
            "amorphous": ["C", "Si", "H", "O"]}
BATCH_KT = 1.0e-2
DENSE_KT = 1.0e-2


def listed():
    return [
        # a fragment of a few atoms, as in force-field fitting or a QM/MM region: pure latency
        dict(name="cluster8", kind="point", recipe="cluster", size=8, iters=10),
        # the parity-sized cluster (216 atoms, about 570 orbitals): an ordinary MD step
        dict(name="cluster216", kind="point", recipe="cluster", size=216, iters=5),
        # liquid water, 300 molecules in a periodic box (1800 orbitals)
        dict(name="water300", kind="point", recipe="water", size=300, iters=3),
        # a 1728-atom periodic solid (about 6650 orbitals): one iteration and forces
        dict(name="diamond6", kind="point", recipe="diamond", size=6, iters=1),
        # the largest single cell: 2744 atoms, about 10560 orbitals
        dict(name="diamond7", kind="point", recipe="diamond", size=7, iters=1),
        # the FP32 iterations with which a mixed-precision cycle of a 512-atom cell begins
        dict(name="mixed_diamond4", kind="point", recipe="diamond", size=4, iters=2, precision=1),
        # a mixed-precision MD step of a 216-atom cell from the charges of the step before
        dict(name="tail_diamond3", kind="tail", recipe="diamond", size=3, iters=4),
        # a solid with a Gamma-centred 2x2x2 mesh: eight real problems per iteration
        dict(name="kpoints_real", kind="point", recipe="amorphous", size=150, iters=2, mesh="gamma"),
        # the shifted mesh of a small cell: eight complex problems per iteration
        dict(name="kpoints_shifted", kind="point", recipe="amorphous", size=40, iters=2, mesh="shifted"),
        # a handful of molecules (one conformer search), where one workgroup's time is what counts
        dict(name="batch32", kind="batch", size=32, iters=8),
        # a screening batch of many small molecules
        dict(name="batch1000", kind="batch", size=1000, iters=5),
        # a host program's eigensolver and density matrix calls
        dict(name="dense1500", kind="dense", size=1500, field="real"),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["point", "point", "point", "mesh", "mixed", "tail", "batch", "dense"])
    if kind == "point":
        recipe = rng.choice(["cluster", "water", "diamond", "amorphous"])
        size = {"cluster": _logint(rng, 5, 343), "water": _logint(rng, 10, 700),
                "diamond": rng.randint(1, 6), "amorphous": _logint(rng, 20, 300)}[recipe]
        iters = 1 if recipe == "diamond" and size > 5 else rng.randint(1, 3)
        return dict(kind="point", recipe=recipe, size=size, iters=iters)
    if kind == "mesh":
        mesh = rng.choice(["gamma", "shifted"])
        size = _logint(rng, 20, 200 if mesh == "gamma" else 50)
        return dict(kind="point", recipe="amorphous", size=size, iters=rng.randint(1, 2), mesh=mesh)
    if kind == "mixed":
        recipe = rng.choice(["water", "diamond"])
        size = _logint(rng, 20, 500) if recipe == "water" else rng.randint(2, 5)
        return dict(kind="point", recipe=recipe, size=size, iters=rng.randint(1, 3), precision=1)
    if kind == "tail":
        return dict(kind="tail", recipe="diamond", size=rng.randint(2, 3), iters=rng.randint(3, 6))
    if kind == "batch":
        return dict(kind="batch", size=_logint(rng, 4, 1000), iters=rng.randint(2, 8))
    return dict(kind="dense", size=_logint(rng, 20, 2000), field=rng.choice(["real", "real", "complex"]))


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------

def _options(case):
    if case["kind"] == "batch":
        return Options(kT=BATCH_KT, max_scc_iter=case["iters"])
    kT, mix, _ = RECIPES[case["recipe"]]
    opt = Options(kT=kT, mix_param=mix, max_scc_iter=case["iters"])
    if case.get("mesh"):
        shift = 0.25 if case["mesh"] == "shifted" else 0.0
        opt.kpoints = np.array([[0.5 * a, 0.5 * b, 0.5 * c] for a in range(2) for b in range(2)
                                for c in range(2)]) + shift
    return opt


def _geometry(case, seed):
    recipe, size = case["recipe"], case["size"]
    if recipe == "cluster":
        side = max(2, math.ceil(size ** (1.0 / 3.0) - 1e-9))
        # the first `size` sites of the lattice (slabs and rows stay together), jittered by the
        # seed; the composition belongs to the case
        coords = synth.cluster_216(seed, side)[0].coords
        species = synth.cluster_216(0, side)[0].species
        return Geometry(coords[:size].copy(), species[:size].copy(), None)
    if recipe == "diamond":
        return synth.diamond_supercell(size, seed)[0]
    if recipe == "water":
        return synth.water_box(size, seed)[0]
    return synth.amorphous_network(size, seed)[0]


def _molecules(case, seed):
    """The chains of the molecule recipe (their lengths and elements belong to the case), with
    bond lengths and angles distorted by the seed."""
    mols, elements = synth.molecule_batch(case["size"], 3)
    rng = np.random.default_rng(seed)
    mols = [Geometry(m.coords + rng.uniform(-0.05, 0.05, m.coords.shape), m.species, None) for m in mols]
    return mols, synth.make_parameters(elements, 103)[0]


def _params(recipe, seed):
    return synth.make_parameters(ELEMENTS[recipe], seed)[0]


def _dense_inputs(case, seed):
    """Hamiltonian and overlap of an extended-Hueckel chain of s functions: Gaussian overlaps of
    jittered sites, Wolfsberg-Helmholz couplings; with a site-dependent phase for complex ones."""
    n = case["size"]
    rng = np.random.default_rng(seed)
    m = math.ceil(n ** (1.0 / 3.0))
    x = np.array(np.meshgrid(*[np.arange(m)] * 3, indexing="ij")).reshape(3, -1).T[:n] * 2.6
    x = x + rng.uniform(-0.3, 0.3, x.shape)
    q = np.sum(x * x, axis=1)
    s = np.exp(-(q[:, None] + q[None, :] - 2.0 * x @ x.T) / (2.0 * 1.6 ** 2))
    eps = rng.uniform(-0.6, -0.1, n)
    h = 0.875 * s * (eps[:, None] + eps[None, :])
    np.fill_diagonal(s, 1.0)
    np.fill_diagonal(h, eps)
    if case["field"] == "complex":
        ph = np.exp(1j * (x @ rng.uniform(0.1, 0.4, 3)))
        h = h * ph[:, None] * ph.conj()[None, :]
        s = s * ph[:, None] * ph.conj()[None, :]
        h, s = 0.5 * (h + h.conj().T), 0.5 * (s + s.conj().T)
    return h, s


def _moved(geo, seed):
    """The next geometry of a trajectory: every atom moved by about 0.005 bohr."""
    rng = np.random.default_rng([seed, 1])
    return geo.coords + rng.uniform(-0.01, 0.01, geo.coords.shape)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "dense":
        h, s = _dense_inputs(case, seed)
        return dict(case=case, h=np.asfortranarray(h), s=np.asfortranarray(s))
    if kind == "batch":
        mols, params = _molecules(case, seed)
        return dict(case=case, mols=mols, params=params, opt=_options(case))
    geo = _geometry(case, seed)
    params = _params(case["recipe"], RECIPES[case["recipe"]][2])
    opt = _options(case)
    state = dict(case=case, coords=geo.coords, latvecs=geo.latvecs)
    if kind == "tail":
        # the step before, converged as far as a trajectory needs it
        before = api.DftbPlus(params, geo, dataclasses.replace(opt, scc_tol=1.0e-4, max_scc_iter=60))
        before.get_energy()
        state["charges"] = before.get_input_charges()
        before.close()
        state["coords"] = _moved(geo, seed)
        state["calc"] = api.DftbPlus(params, geo, opt, precision=1, refine_below=math.inf,
                                     refine_steps=0, tail_below=1.0e-1, tail_steps=2)
    elif case.get("precision"):
        state["calc"] = api.DftbPlus(params, geo, opt, precision=1, refine_below=1.0e-3,
                                     refine_steps=0, tail_below=1.0e-3, tail_steps=2)
    else:
        state["calc"] = api.DftbPlus(params, geo, opt)
    return state


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------

def _run_dense(st):
    n = st["h"].shape[0]
    cplx = st["case"]["field"] == "complex"
    w, C, L = (api.hegvd if cplx else api.sygvd)(st["h"], st["s"])
    f, ef, ebs, ts, _ = api.efilling(w[None, :], np.ones(1), 0.5 * n, DENSE_KT)
    f = 2.0 * f[0]
    occ = int(np.nonzero(f >= np.finfo(float).eps)[0][-1]) + 1
    if cplx:
        dm, edm = api.dm_cmplx(C, f, occ), api.dm_cmplx(C, f, occ, w)
    else:
        dm, edm = api.dm_real(C, f, occ), api.edm_real(C, f, w, occ)
    return dict(levels=w, fermi=ef, band=2.0 * ebs, entropy=2.0 * ts, dm=np.tril(dm), edm=np.tril(edm), factor=np.tril(L))


def run(st):
    kind = st["case"]["kind"]
    if kind == "dense":
        return _run_dense(st)
    if kind == "batch":
        b = api.MoleculeBatch(st["params"], st["mols"], st["opt"])
        e = b.scc()
        g = b.gradients()
        out = dict(energy=e, charges=np.concatenate(b.charges), gradients=np.concatenate(g))
        b.close()
        return out
    calc = st["calc"]
    calc.set_geometry(st["coords"], st["latvecs"])
    if kind == "tail":
        calc.set_input_charges(st["charges"])
    e = calc.get_energy()
    nk = 8 if st["case"].get("mesh") else 1
    pairs = [calc.get_eigenvalues_k(k) for k in range(nk)]
    levels, filling = (np.concatenate([p[k] for p in pairs]) for k in (0, 1))
    return dict(energy=e, charges=calc.get_gross_charges(), gradients=calc.get_gradients(),
                levels=levels, filling=filling, populations=calc.get_orbital_populations())


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------

def _sizes(case):
    """Atoms and orbitals of a point case, by the recipes' compositions."""
    recipe, size = case["recipe"], case["size"]
    if recipe == "water":
        return 3 * size, 6 * size
    if recipe == "diamond":
        nat = 8 * size ** 3
        return nat, 4 * nat - 3 * (int(round(0.1 * nat)) // 2)
    if recipe == "cluster":
        return size, size + 3 * int(round(0.55 * size))
    return size, 4 * size - 3 * int(round(0.05 * size))


def _solve_flops(n, nocc):
    """Reduction, tridiagonalisation and divide and conquer at 4/3 n^3 each, two products of the
    occupied vectors and the density matrix."""
    return 4.0 * n ** 3 + 4.0 * n * n * nocc


def work(case):
    if case["kind"] == "dense":
        n = case["size"]
        c = 2 if case["field"] == "complex" else 1
        flops = c * c * (_solve_flops(n, 0.25 * n) + n ** 3 / 3.0 + 0.25 * n ** 3)
        return dict(bytes=c * 8.0 * n * n * 5 + 8.0 * n, flops=flops)
    if case["kind"] == "batch":
        m, it = case["size"], case["iters"]
        # orbital counts log-uniform in [8, 220]: means of n, n^3
        ln = math.log(220.0 / 8.0)
        n1, n3 = (220 - 8) / ln, (220 ** 3 - 8 ** 3) / (3 * ln)
        nat = n1 / 2.95
        return dict(bytes=8.0 * m * nat * 7, flops=m * n3 * (it * 6.0 + 1.5))
    nat, n = _sizes(case)
    nk = 8 if case.get("mesh") else 1
    c = 4 if case.get("mesh") == "shifted" else 1
    flops = nk * c * (case["iters"] * _solve_flops(n, 0.5 * n) + 1.2 * n ** 3)
    return dict(bytes=8.0 * (3 * nat + nat + 3 * nat + 3 * n), flops=flops)


def tolerance(case):
    # measured: two passes over the same inputs (their atomic sums are in no fixed order) differ by
    # 1e-13 (FP64), 4e-6 (FP32 iterations; 2e-5 from float64) and 1e-6 (tail); FP64 limits leave
    # room for other orthonormal bases of close levels and for the iterations' growth of an error
    if case.get("precision"):
        return {"rel": 1.0e-4, "max": 1.0e-3}
    if case["kind"] == "tail":
        return {"rel": 2.0e-5, "max": 1.0e-4}
    return {"rel": 1.0e-9, "max": 1.0e-8}


# ---------------------------------------------------------------------------------------------
# the same in float64, from the formulas
# ---------------------------------------------------------------------------------------------

def _end_weights():
    """First and second derivative at node 7 of the Lagrange basis of nodes 0..7."""
    out = np.zeros((2, 8))
    for k in range(8):
        p = np.poly1d([1.0])
        for m in range(8):
            if m != k:
                p = p * np.poly1d([1.0, -m]) / (k - m)
        out[:, k] = p.deriv(1)(7.0), p.deriv(2)(7.0)
    return torch.tensor(out)


_END = _end_weights()


def _lagrange(table, dist, r):
    """Slater-Koster integrals at distances r: degree-7 polynomial through the eight grid rows
    around r, beyond the grid a quintic that joins with value, slope and curvature and ends at 0."""
    rows = table.shape[0]
    rmax = rows * dist + 1.0
    nodes = torch.arange(8, dtype=torch.float64)

    def weights(t):
        """Lagrange weights of nodes 0..7 at t."""
        out = []
        for k in range(8):
            num = torch.ones_like(t)
            for m in range(8):
                if m != k:
                    num = num * (t - nodes[m]) / float(k - m)
            out.append(num)
        return torch.stack(out, dim=1)

    ind = torch.floor(r.detach() / dist).long()
    last = torch.clamp(torch.minimum(ind + 4, torch.tensor(rows)), min=8)
    inside = ind < rows
    idx = last[:, None] - 8 + torch.arange(8)[None, :]
    t = r / dist - (last - 7).to(torch.float64)
    grid = torch.einsum("pk,pkc->pc", weights(torch.where(inside, t, torch.zeros_like(t))), table[idx])
    # value and derivatives of the last polynomial at the last row (node 7)
    tail = table[rows - 8:]
    y0, y1, y2 = tail[7], (_END[0] @ tail) / dist, (_END[1] @ tail) / dist ** 2
    # rises from the end of the range (u = 0) to the grid end (u = 1), du/dr = -1
    u = (rmax - r)[:, None]
    a, b = -y1, y2
    quintic = ((6 * y0 - 3 * a + 0.5 * b) * u ** 2 + (-15 * y0 + 7 * a - b) * u + (10 * y0 - 4 * a + 0.5 * b)) * u ** 3
    inside = inside[:, None]
    return torch.where(inside, grid, torch.where((r < rmax)[:, None], quintic, torch.zeros_like(quintic)))


def _blocks(sk, sh1, sh2, u):
    """Diatomic blocks (pairs, orbitals of atom 2, orbitals of atom 1), p order y, z, x."""
    v = u[:, [1, 2, 0]]
    cols, k = [], 0
    for l1 in sh1:
        rows = []
        for l2 in sh2:
            if l1 == 0 and l2 == 0:
                rows.append(sk[:, k, None, None])
            elif l1 + l2 == 1:
                e = v * sk[:, k, None]
                rows.append(e[:, :, None] if l1 == 0 else -e[:, None, :])
            else:
                s, p = sk[:, k, None, None], sk[:, k + 1, None, None]
                rows.append((s - p) * v[:, :, None] * v[:, None, :] + p * torch.eye(3, dtype=torch.float64))
            k += min(l1, l2) + 1
        cols.append(torch.cat(rows, dim=1))
    return torch.cat(cols, dim=2)


def _short_gamma(r, ua, ub):
    """Difference between 1/r and the interaction of two exponential charges."""
    ta, tb = 3.2 * ua, 3.2 * ub
    if abs(ua - ub) < 1e-10:
        t = ta
        return torch.exp(-t * r) * (1 / r + 0.6875 * t + 0.1875 * t * t * r + t ** 3 * r * r / 48.0)

    def part(x, y):
        d = x * x - y * y
        return torch.exp(-x * r) * (0.5 * y ** 4 * x / d ** 2 - (y ** 6 - 3 * y ** 4 * x * x) / (r * d ** 3))
    return part(ta, tb) + part(tb, ta)


def _onsite_gamma(ua, ub):
    ta, tb = 3.2 * ua, 3.2 * ub
    return 0.5 * (ua + ub) if abs(ua - ub) < 1e-10 else 0.5 * (ta * tb / (ta + tb) + (ta * tb) ** 2 / (ta + tb) ** 3)


def _repulsive(rep, r):
    xs = torch.tensor(rep.xstart)
    e = torch.zeros_like(r)
    a1, a2, a3 = rep.expcoeffs
    e = torch.where(r < xs[0], torch.exp(-a1 * r + a2) + a3, e)
    for m in range(len(rep.xstart)):
        hi = rep.cutoff if m + 1 == len(rep.xstart) else float(xs[m + 1])
        c = rep.spcoeffs[m] if m + 1 < len(rep.xstart) else rep.lastcoeffs
        d, p = r - xs[m], torch.zeros_like(r)
        for x in c[::-1]:
            p = p * d + float(x)
        e = torch.where((r >= xs[m]) & (r < hi), p, e)
    return e


class _System:
    """Pair lists and, for coordinates X, the sparse H0 and S blocks, gamma and repulsive energy."""

    def __init__(self, params, coords, species, lat):
        self.p, self.species, self.lat = params, species, lat
        nat = len(species)
        self.nat = nat
        self.norb = np.array([params.species[s].norb for s in species])
        self.off = np.concatenate([[0], np.cumsum(self.norb)])
        self.q0 = np.array([float(sum(params.species[s].occ)) for s in species])
        self.cut = max(params.nrows * params.dist + 1.0, 30.0)
        cells = np.zeros((1, 3))
        if lat is not None:
            # exp(-3.2 U r) falls below 1e-12 within 30 bohr for U >= 0.3
            n = [int(math.ceil(self.cut * np.linalg.norm(np.linalg.inv(lat)[:, k]))) for k in range(3)]
            cells = np.array([[a, b, c] for a in range(-n[0], n[0] + 1) for b in range(-n[1], n[1] + 1)
                              for c in range(-n[2], n[2] + 1)], dtype=float)
        rows = []
        for c in cells:
            T = c @ lat if lat is not None else np.zeros(3)
            d = coords[None, :, :] + T - coords[:, None, :]
            r2 = np.sum(d * d, axis=2)
            i, j = np.nonzero(r2 <= self.cut ** 2)
            keep = (j > i) | ((j == i) & (r2[i, j] > 1e-12))
            rows.append((i[keep], j[keep], np.tile(c, (int(keep.sum()), 1))))
        self.i, self.j = (np.concatenate([r[k] for r in rows]) for k in (0, 1))
        self.cell = np.concatenate([r[2] for r in rows])
        self.shift = torch.tensor(self.cell @ lat if lat is not None else 0.0 * self.cell)

    def vectors(self, X):
        v = X[self.j] + self.shift - X[self.i]
        return v, torch.sqrt(torch.sum(v * v, dim=1))

    def h0s(self, X):
        """[(i, j, pair index, H0 block, S block)] per ordered species pair, rows on atom j."""
        v, r = self.vectors(X)
        rmax = self.p.nrows * self.p.dist + 1.0
        near = (r.detach() < rmax).numpy()
        out = []
        for a in range(self.p.nspecies):
            for b in range(self.p.nspecies):
                k = np.nonzero(near & (self.species[self.i] == a) & (self.species[self.j] == b))[0]
                if len(k) == 0:
                    continue
                u = v[k] / r[k][:, None]
                sh = self.p.species[a].shells, self.p.species[b].shells
                h, s = (_blocks(_lagrange(torch.tensor(t[(a, b)]), self.p.dist, r[k]), *sh, u)
                        for t in (self.p.ham, self.p.over))
                out.append((k, h, s))
        return out

    def index(self, k):
        """Dense rows (orbitals of j) and columns (orbitals of i) of blocks k (one species pair)."""
        rows = self.off[self.j[k]][:, None, None] + np.arange(self.norb[self.j[k[0]]])[None, :, None]
        cols = self.off[self.i[k]][:, None, None] + np.arange(self.norb[self.i[k[0]]])[None, None, :]
        return np.broadcast_arrays(rows, cols)

    def dense(self, blocks, which, diag, phase=None):
        """Full Hermitian matrix; blocks of an atom with its own images come in +T, -T pairs."""
        n = int(self.off[-1])
        m = np.zeros((n, n), dtype=float if phase is None else complex)
        for blk in blocks:
            r, c = self.index(blk[0])
            x = blk[which].detach().numpy()
            x = x if phase is None else x * phase[blk[0]][:, None, None]
            other = self.i[blk[0]] != self.j[blk[0]]
            np.add.at(m, (r, c), x)
            np.add.at(m, (c[other], r[other]), x[other].conj())
        m[np.arange(n), np.arange(n)] += diag
        return m

    def onsite(self):
        return np.concatenate([[self.p.species[s].onsite[k] for k in self.p.species[s].orb_shell()]
                               for s in self.species])

    def gamma(self, X):
        nat = self.nat
        v, r = self.vectors(X)
        hub = [s.hubbu[0] for s in self.p.species]
        if self.lat is None:
            g = torch.zeros(nat * nat, dtype=torch.float64)
            long = 1.0 / torch.sqrt(torch.sum((X[:, None] - X[None]) ** 2, dim=2) + torch.eye(nat, dtype=torch.float64))
            g = g + (long - torch.eye(nat, dtype=torch.float64)).reshape(-1)
        else:
            g = self._ewald(X, v, r).reshape(-1)
        idx, val = [], []
        for a in range(self.p.nspecies):
            for b in range(self.p.nspecies):
                k = np.nonzero((self.species[self.i] == a) & (self.species[self.j] == b))[0]
                if len(k):
                    idx.append(k)
                    val.append(_short_gamma(r[k], hub[a], hub[b]))
        if idx:
            g = g.index_add(0, torch.tensor(self._pair(np.concatenate(idx))), -torch.cat(val))
            k = np.concatenate(idx)
            o = self.i[k] != self.j[k]
            g = g.index_add(0, torch.tensor(self.j[k][o] * nat + self.i[k][o]), -torch.cat(val)[o])
        u = torch.tensor([_onsite_gamma(hub[s], hub[s]) for s in self.species])
        return g.reshape(nat, nat) + torch.diag(u)

    def _pair(self, k):
        return self.i[k] * self.nat + self.j[k]

    def _ewald(self, X, v, r):
        """1/R summed over the lattice: real-space part over the pair list, reciprocal part to 1e-16."""
        nat = self.nat
        vol = abs(np.linalg.det(self.lat))
        al = 6.0 / self.cut
        rec = 2.0 * math.pi * np.linalg.inv(self.lat).T
        gmax = 2.0 * al * 6.2
        n = [int(math.ceil(gmax * np.linalg.norm(self.lat[k]) / (2 * math.pi))) for k in range(3)]
        G = np.array([[a, b, c] for a in range(-n[0], n[0] + 1) for b in range(-n[1], n[1] + 1)
                      for c in range(-n[2], n[2] + 1) if (a, b, c) > (0, 0, 0)], dtype=float) @ rec
        G = torch.tensor(G[np.sum(G * G, axis=1) <= gmax ** 2].reshape(-1, 3))
        g2 = torch.sum(G * G, dim=1)
        w = 8.0 * math.pi / vol * torch.exp(-g2 / (4 * al * al)) / g2
        ph = X @ G.T
        c, s = torch.cos(ph), torch.sin(ph)
        m = ((c * w) @ c.T + (s * w) @ s.T - math.pi / (vol * al * al)
             - 2.0 * al / math.sqrt(math.pi) * torch.eye(nat, dtype=torch.float64)).reshape(-1)
        e = torch.erfc(al * r) / r
        m = m.index_add(0, torch.tensor(self._pair(np.arange(len(self.i)))), e)
        o = np.nonzero(self.i != self.j)[0]
        return m.index_add(0, torch.tensor(self.j[o] * nat + self.i[o]), e[o]).reshape(nat, nat)

    def repulsive(self, X):
        _, r = self.vectors(X)
        e = torch.zeros((), dtype=torch.float64)
        for a in range(self.p.nspecies):
            for b in range(self.p.nspecies):
                rep = self.p.rep[(a, b)]
                k = np.nonzero((r.detach().numpy() < rep.cutoff) & (self.species[self.i] == a)
                               & (self.species[self.j] == b))[0]
                if len(k):
                    half = torch.tensor(np.where(self.i[k] == self.j[k], 0.5, 1.0))
                    e = e + torch.sum(half * _repulsive(rep, r[k]))
        return e


def _fermi(eig, weights, nel, kT):
    """Fillings (two electrons per level), entropy TS; mu by bisection of the electron count."""
    lo, hi = eig.min() - 1.0, eig.max() + 1.0
    f = np.ones_like(eig)
    for _ in range(200):
        mu = 0.5 * (lo + hi)
        f = 1.0 / (1.0 + np.exp(np.clip((eig - mu) / kT, -700, 700)))
        if 2.0 * float(np.sum(weights[:, None] * f)) > nel:
            hi = mu
        else:
            lo = mu
    if nel >= 2 * eig.shape[1] - 1e-9:
        f = np.ones_like(eig)
    mid = (f > 1e-300) & (f < 1.0)
    x = np.where(mid, f, 0.5)
    ent = np.where(mid, x * np.log(x) + (1 - x) * np.log1p(-x), 0.0)
    return 2.0 * f, -2.0 * kT * float(np.sum(weights[:, None] * ent))


def _broyden(history, q, diff, alpha):
    """Johnson's modified Broyden step over the differences of all iterations so far."""
    history.append((q.copy(), diff.copy()))
    new = q + alpha * diff
    m = len(history) - 1
    if m == 0:
        return new
    dF, u = [], []
    for k in range(m):
        d = history[k + 1][1] - history[k][1]
        norm = max(np.linalg.norm(d), np.finfo(float).eps)
        dF.append(d / norm)
        u.append(alpha * d / norm + (history[k + 1][0] - history[k][0]) / norm)
    w = np.array([max(1.0, min(1.0e5, 1.0e-2 / max(np.linalg.norm(history[k + 1][1]), 1e-300))) for k in range(m)])
    A = np.array(dF)
    beta = w[:, None] * w[None, :] * (A @ A.T) + 1.0e-4 * np.eye(m)
    coef = np.linalg.solve(beta.T, w * (A @ diff))
    return new - (w * coef) @ np.array(u)


def _scc(params, coords, species, lat, opt, charges=None):
    sys_ = _System(params, coords, species, lat)
    X = torch.tensor(coords, requires_grad=True)
    n, off = int(sys_.off[-1]), sys_.off
    gamma = sys_.gamma(X).detach().numpy()
    blocks = sys_.h0s(X)
    kpts = opt.kpoints
    phases = [None] if kpts is None else [np.exp(2j * np.pi * (sys_.cell @ k)) for k in kpts]
    wk = np.full(len(phases), 1.0 / len(phases))
    H0 = [sys_.dense(blocks, 1, sys_.onsite(), ph) for ph in phases]
    S = [sys_.dense(blocks, 2, 1.0, ph) for ph in phases]
    chol = [np.linalg.inv(np.linalg.cholesky(s)) for s in S]
    owner = np.repeat(np.arange(sys_.nat), sys_.norb)
    nel = float(sys_.q0.sum())
    q = sys_.q0.copy() if charges is None else charges.copy()
    history = []
    for it in range(opt.max_scc_iter):
        pot = (gamma @ (q - sys_.q0))[owner]
        eig, vec = [], []
        for h0, s, li in zip(H0, S, chol):
            h = h0 + 0.5 * s * (pot[:, None] + pot[None, :])
            e, z = np.linalg.eigh(li @ h @ li.conj().T)
            eig.append(e)
            vec.append(li.conj().T @ z)
        eig = np.array(eig)
        f, ts = _fermi(eig, wk, nel, max(opt.kT, 1e-8))
        rho = [wk[k] * (c * f[k]) @ c.conj().T for k, c in enumerate(vec)]
        pop = sum(np.sum(r * s.conj(), axis=1).real for r, s in zip(rho, S))
        qout = np.add.reduceat(pop, off[:-1])
        diff = qout - q
        if np.max(np.abs(diff)) < opt.scc_tol:
            break
        if it + 1 < opt.max_scc_iter:
            q = _broyden(history, q, diff, opt.mix_param)
    dq = qout - sys_.q0
    shift = gamma @ dq
    e_h0 = sum(float(np.sum(r * h.conj()).real) for r, h in zip(rho, H0))
    erep = sys_.repulsive(X)
    energy = e_h0 + 0.5 * float(dq @ shift) + erep.item() - ts
    # gradient of the energy functional at fixed density, energy-weighted density and charges
    wden = [wk[k] * (c * (f[k] * eig[k])) @ c.conj().T for k, c in enumerate(vec)]
    sh = torch.tensor(shift)
    tdq = torch.tensor(dq)
    func = 0.5 * tdq @ (sys_.gamma(X) @ tdq) + erep
    for k, h, s in blocks:
        r, c = sys_.index(k)
        rb = sum((m[r, c].conj() * (1.0 if ph is None else ph[k][:, None, None])).real for m, ph in zip(rho, phases))
        wb = sum((m[r, c].conj() * (1.0 if ph is None else ph[k][:, None, None])).real for m, ph in zip(wden, phases))
        rb, wb = torch.tensor(rb), torch.tensor(wb)
        v = 0.5 * (sh[sys_.i[k]] + sh[sys_.j[k]])[:, None, None]
        func = func + 2.0 * torch.sum(rb * h + (rb * v - wb) * s)
    grad = torch.autograd.grad(func, X)[0].numpy()
    return dict(energy=energy, charges=-dq, gradients=grad, levels=eig.reshape(-1), filling=f.reshape(-1), populations=pop)


def _seconds(n, solves, complex_):
    """Rough time of that many eigensolutions on a few cores."""
    return solves * (n / 1000.0) ** 3 * (1.5 if complex_ else 0.5)


def exact(case, seed):
    kind = case["kind"]
    if kind == "dense":
        h, s = _dense_inputs(case, seed)
        n = case["size"]
        L = np.linalg.cholesky(s)
        li = np.linalg.inv(L)
        w, z = np.linalg.eigh(li @ h @ li.conj().T)
        C = li.conj().T @ z
        f, ts = _fermi(w[None, :], np.ones(1), float(n), DENSE_KT)
        f = f[0]
        dm, edm = ((C * x) @ C.conj().T for x in (f, f * w))
        return dict(levels=w, fermi=None, band=float(f @ w), entropy=ts, dm=np.tril(dm), edm=np.tril(edm), factor=L)
    opt = _options(case)
    if kind == "batch":
        if case["size"] > 200:
            return None
        mols, params = _molecules(case, seed)
        got = [_scc(params, m.coords, m.species, None, opt) for m in mols]
        return dict(energy=np.array([g["energy"] for g in got]),
                    charges=np.concatenate([g["charges"] for g in got]),
                    gradients=np.concatenate([g["gradients"] for g in got]))
    # the tail's converged start costs a whole cycle, and mixed precision has no float64 path of
    # its own: its FP32 iterations are compared with the same iterations in float64
    nat, n = _sizes(case)
    solves = case["iters"] * (8 if case.get("mesh") else 1)
    if kind == "tail" or _seconds(n, solves, bool(case.get("mesh"))) > 12.0:
        return None
    geo = _geometry(case, seed)
    return _scc(_params(case["recipe"], RECIPES[case["recipe"]][2]), geo.coords, geo.species, geo.latvecs, opt)
