"""The work that programs have this engine do, as cases that can be timed and compared.

Each case goes through the public Python entry points: Fock builds of one molecule (Context.contract_jk) and of a
resident set (Batch), whole RHF solves alone (scf_rhf) and served together (Server), the nuclear gradient, density-fitted
J and K in the three exchange precisions (DfTensor) and a density-fitted solve (df_rhf).  The molecules are the
framework's own workloads: water clusters on a lattice and all-trans alkanes, displaced a little by the seed.

exact() is an independent evaluation in 64 bits: Hermite (McMurchie-Davidson) integrals written in plain torch.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch


def _load():
    """The package: its folder's name has a hyphen, so it is imported by its place."""
    if "hf_rs_amd" not in sys.modules:
        folder = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hf-rs_amd")
        spec = importlib.util.spec_from_file_location("hf_rs_amd", os.path.join(folder, "__init__.py"),
                                                      submodule_search_locations=[folder])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["hf_rs_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["hf_rs_amd"]


hf = _load()
from hf_rs_amd import molecules as M  # noqa: E402

JKFIT = "def2-universal-jkfit"
AUX = {"cc-pvdz": JKFIT, "def2-svp": "def2-svp-rifit"}


def listed():
    return [
        # a Fock build of the smallest molecule in earnest use: latency and launches
        {"name": "jk_water_631gs", "path": "jk", "mol": "water", "m": 1, "basis": "6-31g*"},
        # an ordinary Fock build, generally contracted basis
        {"name": "jk_water4_ccpvdz", "path": "jk", "mol": "water", "m": 4, "basis": "cc-pvdz"},
        # the direct Fock build of (H2O)16 / cc-pVDZ, the single-molecule headline
        {"name": "jk_water16_ccpvdz", "path": "jk", "mol": "water", "m": 16, "basis": "cc-pvdz"},
        # fused Fock builds of a resident set of mixed molecules, the batched headline's unit of work
        {"name": "batch96_def2svp", "path": "batch", "count": 96, "basis": "def2-svp"},
        # served solves with builds of the density change: the batched headline's serving form
        {"name": "server40_def2svp", "path": "server", "count": 40, "basis": "def2-svp", "incremental": True},
        # one whole RHF solve with the reference's algorithm (full builds)
        {"name": "scf_water8_ccpvdz", "path": "scf", "mol": "water", "m": 8, "basis": "cc-pvdz", "incremental": False},
        # a geometry optimiser's gradient
        {"name": "grad_octane_631g", "path": "grad", "mol": "alkane", "m": 8, "basis": "6-31g"},
        # a whole density-fitted solve: factors, builds, eigensolver
        {"name": "df_rhf_water6_ccpvdz", "path": "df_rhf", "mol": "water", "m": 6, "basis": "cc-pvdz",
         "precision": "fp64"},
        # density-fitted J and K from factors in memory, FP64, an ordinary large molecule
        {"name": "df_fp64_water32_ccpvdz", "path": "df", "mol": "water", "m": 32, "basis": "cc-pvdz",
         "precision": "fp64"},
        # the same with FP32 exchange, a medium molecule
        {"name": "df_fp32_water20_ccpvdz", "path": "df", "mol": "water", "m": 20, "basis": "cc-pvdz",
         "precision": "fp32"},
        # the same with split-BF16 exchange
        {"name": "df_bf16x3_water32_ccpvdz", "path": "df", "mol": "water", "m": 32, "basis": "cc-pvdz",
         "precision": "bf16x3"},
        # the largest: factors that are kept packed (n 1200, rank 6384, 240 occupied)
        {"name": "df_fp64_water48_ccpvdz", "path": "df", "mol": "water", "m": 48, "basis": "cc-pvdz",
         "precision": "fp64"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    path = rng.choice(["jk", "jk", "batch", "server", "scf", "grad", "df", "df", "df", "df_rhf"])
    mol = rng.choice(["water", "alkane"])
    c = {"path": path}
    if path == "jk":
        basis = rng.choice(["sto-3g", "6-31g*", "def2-svp", "cc-pvdz"])
        c.update(mol=mol, m=_log_int(rng, 1, 16 if mol == "water" else 12), basis=basis)
    elif path == "batch":
        c.update(count=_log_int(rng, 4, 96), basis=rng.choice(["def2-svp", "6-31g*"]))
    elif path == "server":
        c.update(count=_log_int(rng, 2, 32), basis=rng.choice(["def2-svp", "6-31g*"]),
                 incremental=rng.random() < 0.5)
    elif path == "scf":
        c.update(mol=mol, m=_log_int(rng, 1, 8 if mol == "water" else 6),
                 basis=rng.choice(["sto-3g", "6-31g*", "def2-svp", "cc-pvdz"]), incremental=rng.random() < 0.5)
    elif path == "grad":
        c.update(mol=mol, m=_log_int(rng, 1, 8), basis=rng.choice(["sto-3g", "6-31g"]))
    elif path == "df":
        basis = rng.choice(["cc-pvdz", "cc-pvdz", "def2-svp"])
        top = 32 if mol == "water" else 12
        c.update(mol=mol, m=_log_int(rng, 2, top), basis=basis, precision=rng.choice(["fp64", "fp32", "bf16x3"]))
    else:
        c.update(mol=mol, m=_log_int(rng, 1, 6), basis=rng.choice(["cc-pvdz", "def2-svp"]),
                 precision=rng.choice(["fp64", "fp64", "bf16x3"]))
    c["shake"] = rng.randrange(1, 1 << 20)  # two draws of one size are still two geometries or sets
    return c


# ---- inputs ----

def _shaken(mol, rng):
    """The molecule with every atom displaced by about 0.02 A, as along a trajectory."""
    xyz = mol.xyz + rng.standard_normal(mol.xyz.shape) * 0.02 * M.ANGSTROM_TO_BOHR
    return M.Molecule(mol.symbols, xyz, name=mol.name)


def _rng(case, seed):
    return np.random.Generator(np.random.PCG64([int(seed) % (1 << 32), int(case.get("shake", 0))]))


def _molecule(case, rng):
    if case["mol"] == "alkane":
        return _shaken(M.alkane(case["m"]), rng)
    return _shaken(M.water_cluster_m(case["m"], seed=int(rng.integers(0, 1 << 31))), rng)


def _basis(name, mol):
    return hf.Basis.from_g94(M.basis_text(name), mol.symbols, mol.xyz)


def _orbitals(n, o, rng):
    """o orthonormal columns: occupied orbitals of an orthonormal basis."""
    q, _ = np.linalg.qr(rng.standard_normal((n, o)))
    return np.ascontiguousarray(q)


def _set(case, rng):
    """Half alkanes C1..C12, half water clusters of 1..8, as the batched workload: which ones is the case's, their
    geometries are the seed's."""
    sizes = np.random.Generator(np.random.PCG64([3, int(case.get("shake", 0))]))
    mols = []
    for i in range(case["count"]):
        if i % 2 == 0:
            mols.append(_shaken(M.alkane(int(sizes.integers(1, 13))), rng))
        else:
            mols.append(_shaken(M.water_cluster_m(int(sizes.integers(1, 9)), seed=int(rng.integers(0, 1 << 31))), rng))
    return mols


def _molecules(case):
    """The molecules that work() prices."""
    rng = _rng(case, 1)
    return _set(case, rng) if "count" in case else [_molecule(case, rng)]


def prepare(case, seed):
    rng = _rng(case, seed)
    path = case["path"]
    if path in ("batch", "server"):
        mols = _set(case, rng)
        bases = [_basis(case["basis"], m) for m in mols]
        if path == "server":
            return {"case": case, "mols": mols, "bases": bases}
        batch = hf.Batch(bases)
        dens = []
        for i, (m, b) in enumerate(zip(mols, bases)):
            c = _orbitals(b.n, m.n_electrons() // 2, rng)
            dens.append(2.0 * c @ c.T)
            batch.set_density(i, dens[-1])
        return {"case": case, "mols": mols, "bases": bases, "batch": batch, "dens": dens}
    mol = _molecule(case, rng)
    basis = _basis(case["basis"], mol)
    o = mol.n_electrons() // 2
    s = {"case": case, "mol": mol, "basis": basis}
    if path == "jk":
        c = _orbitals(basis.n, o, rng)
        s.update(ctx=hf.Context(basis), p=2.0 * c @ c.T)
    elif path == "grad":
        c = _orbitals(basis.n, o, rng)
        eps = -np.sort(rng.uniform(0.3, 20.0, o))[::-1]
        s.update(ctx=hf.Context(basis), p=2.0 * c @ c.T, w=2.0 * (c * eps) @ c.T)
    elif path == "df":
        aux = _basis(AUX[case["basis"]], mol)
        s.update(aux=aux, df=hf.DfTensor(basis, aux), c=_orbitals(basis.n, o, rng))
    elif path == "df_rhf":
        s.update(aux=_basis(AUX[case["basis"]], mol))
    return s


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "jk":
        return state["ctx"].contract_jk(state["p"])
    if path == "batch":
        b = state["batch"]
        b.jk()
        out = [b.get_jk(i) for i in range(len(state["bases"]))]
        return np.concatenate([j.ravel() for j, _ in out]), np.concatenate([k.ravel() for _, k in out])
    if path == "server":
        srv = hf.Server(capacity=len(state["bases"]))
        ids = [srv.submit([b], [m.zxyz], keep_density=True, incremental=case["incremental"])
               for b, m in zip(state["bases"], state["mols"])]
        srv.run()
        res = [srv.result(i, density=True) for i in ids]
        srv.close()
        return {"energy": np.array([r["steps_result"][0]["energy"] for r in res]),
                "density": np.concatenate([r["density"].ravel() for r in res])}
    if path == "scf":
        r = hf.scf_rhf(state["basis"], state["mol"].zxyz, want_matrices=True, incremental=case["incremental"])
        return {"energy": r["total_energy"], "density": r["density"], "fock": r["fock"]}
    if path == "grad":
        return state["ctx"].rhf_gradient(state["mol"].zxyz, state["p"], state["w"])
    if path == "df":
        j, k, _ = state["df"].jk_precision(state["c"], case["precision"])
        return j, k
    r = hf.df_rhf(state["basis"], state["aux"], state["mol"].zxyz, k_precision=case["precision"])
    return {"energy": r["total_energy"], "density": r["density"], "fock": r["fock"]}


# ---- what a pass cannot do without ----

def _jk_flops(basis):
    """A lower count for one direct build: for each surviving quartet of functions the six updates of J and K (12), and
    for each primitive quartet of the surviving shell quartets 60 for the pair distance, the Boys function and one
    recurrence step.  Survival by overlap: pairs with exp(-mu R^2) below 1e-10 fall out."""
    a = basis.a
    first, dims, expo = [], [], []
    for f in range(basis.n):
        lx = a["lxyz"][f]
        if lx[1] == 0 and lx[2] == 0:
            first.append(f)
            dims.append((lx[0] + 1) * (lx[0] + 2) // 2)
            expo.append(a["exponent"][a["prim_offset"][f]:a["prim_offset"][f + 1]])
    centre = a["center"][first]
    r2 = ((centre[:, None] - centre[None]) ** 2).sum(-1)
    small = np.array([e.min() for e in expo])
    npr = np.array([len(e) for e in expo], float)
    dims = np.array(dims, float)
    iu = np.tril_indices(len(first))
    mu = (small[:, None] * small[None] / (small[:, None] + small[None]))[iu]
    keep = mu * r2[iu] < 23.0
    screen = np.exp(-mu * r2[iu])[keep]
    order = np.argsort(-screen)
    screen = screen[order]
    f2 = np.outer(dims, dims)[iu][keep][order]
    p2 = np.minimum(np.outer(npr, npr)[iu][keep][order], 9.0)
    reach = np.searchsorted(-screen, -1e-10 / screen, side="right")
    funcs = 0.5 * (f2 * np.concatenate([[0.0], np.cumsum(f2)])[reach]).sum()
    prims = 0.5 * (p2 * np.concatenate([[0.0], np.cumsum(p2)])[reach]).sum()
    return 12.0 * funcs + 60.0 * prims


def work(case):
    path = case["path"]
    mols = _molecules(case)
    bases = [_basis(case["basis"], m) for m in mols]
    nn = float(sum(b.n * b.n for b in bases))
    if path in ("jk", "batch"):
        return {"bytes": 24.0 * nn, "flops": sum(_jk_flops(b) for b in bases)}
    if path in ("server", "scf"):
        # no fewer than eight builds' iterations converge; builds of the density change count as two full ones
        builds = 2 if case["incremental"] else 8
        cube = float(sum(float(b.n) ** 3 for b in bases))
        return {"bytes": 24.0 * 8 * nn, "flops": builds * sum(_jk_flops(b) for b in bases) + 8 * 20 * cube}
    if path == "grad":
        return {"bytes": 16.0 * nn + 24.0 * len(mols[0].symbols), "flops": 4.0 * _jk_flops(bases[0])}
    aux = float(_basis(AUX[case["basis"]], mols[0]).n)
    n, o = float(bases[0].n), mols[0].n_electrons() / 2.0
    jk = 2.0 * aux * n * n * o + n * n * aux * o + 2.0 * aux * n * n
    if path == "df":
        return {"bytes": aux * n * (n + 1) / 2 * 8.0 + 8.0 * n * o + 16.0 * n * n, "flops": jk}
    return {"bytes": 10 * aux * n * (n + 1) / 2 * 8.0, "flops": aux * aux * n * n + 10 * (jk + 20 * n ** 3)}


def tolerance(case):
    if case["path"] in ("jk", "batch"):
        return {"rel": 1e-12, "max": 1e-10}  # 3.2e-13 against exact(): the Schwarz screening at 1e-12
    if case["path"] == "grad":
        return {"rel": 1e-11, "max": 1e-9}
    if case["path"] in ("server", "scf", "df_rhf"):
        return {"rel": 1e-8, "max": 1e-6}  # where the iterations stop, not what a sum's order does
    # against exact(): 7e-12 (the metric's small eigenvalues), 2.4e-7 and 1.7e-6
    return {"fp64": {"rel": 3e-11, "max": 3e-9}, "fp32": {"rel": 1e-6, "max": 1e-4},
            "bf16x3": {"rel": 7e-6, "max": 7e-4}}[case["precision"]]


# ---- the same in plain torch, 64 bits ----

class _Boys(torch.autograd.Function):
    """F_0 .. F_m of T, stacked on a new first axis; dF_n/dT = -F_{n+1}."""

    @staticmethod
    def forward(ctx, t, m):
        top = m + 1
        f = torch.empty((top + 1,) + t.shape, dtype=t.dtype, device=t.device)
        far = t > 40.0
        ts = torch.where(far, torch.ones_like(t), t)
        # F_top by its ascending series, the others by downward recursion
        term = torch.full_like(ts, 1.0 / (2 * top + 1))
        total = term.clone()
        for k in range(1, 170):
            term = term * (2.0 * ts / (2 * top + 2 * k + 1))
            total += term
        ex = torch.exp(-ts)
        f[top] = ex * total
        for n in range(top - 1, -1, -1):
            f[n] = (2.0 * ts * f[n + 1] + ex) / (2 * n + 1)
        # far: erf is one to the last bit, upward recursion is stable
        tf = torch.where(far, t, torch.full_like(t, 50.0))
        g = 0.5 * torch.sqrt(math.pi / tf)
        exf = torch.exp(-tf)
        for n in range(top + 1):
            f[n] = torch.where(far, g, f[n])
            g = ((2 * n + 1) * g - exf) / (2.0 * tf)
        ctx.save_for_backward(f)
        return f[:top]

    @staticmethod
    def backward(ctx, grad):
        (f,) = ctx.saved_tensors
        return -(grad * f[1:]).sum(0), None


def _powers(l):
    return [(x, y, l - x - y) for x in range(l, -1, -1) for y in range(l - x, -1, -1)]


def _hermites(l):
    return [h for d in range(l + 1) for h in _powers(d)]


class _Shells:
    """Shells of a basis: primitives, functions and component factors, from the flat arrays."""

    def __init__(self, basis, xyz, device):
        a = basis.a
        self.n = basis.n
        self.rows = []  # (l, atom, first function, exponents, coefficients, component factors)
        f = 0
        while f < basis.n:
            l = int(a["lxyz"][f].sum())
            nf = (l + 1) * (l + 2) // 2
            sl = slice(a["prim_offset"][f], a["prim_offset"][f + 1])
            coef = a["coefficient"][sl]
            fac = [float(a["coefficient"][a["prim_offset"][f + i]] / coef[0]) for i in range(nf)]
            order = [_powers(l).index(tuple(int(v) for v in a["lxyz"][f + i])) for i in range(nf)]
            self.rows.append((l, int(a["atom_index"][f]), f, a["exponent"][sl], coef, fac, order))
            f += nf
        self.xyz, self.device = xyz, device

    def prims(self):
        """By l: (shell's first function, atom, exponent, coefficient) of every primitive shell."""
        out = {}
        for l, at, f, ex, co, _, _ in self.rows:
            out.setdefault(l, []).extend((f, at, e, c) for e, c in zip(ex, co))
        return out

    def factors(self):
        """Per function its component factor, and where its component stands in _powers order."""
        fac = torch.ones(self.n, dtype=torch.float64, device=self.device)
        slot = np.zeros(self.n, np.int64)
        for l, _, f, _, _, fc, order in self.rows:
            for i in range(len(fc)):
                fac[f + i] = fc[i]
                slot[f + i] = f + order[i]
        return fac, torch.as_tensor(slot, device=self.device)


def _expansion(la, lb, a, b, ab, extra=0):
    """One-axis Hermite coefficients E[i][j][t], i <= la, j <= lb + extra, of primitive pairs, without exp(-mu R^2)."""
    p = a + b
    xpa, xpb = -b / p * ab, a / p * ab
    h = 0.5 / p
    one = torch.ones_like(p)
    e = {(0, 0): [one]}

    def at(v, t):
        return v[t] if 0 <= t < len(v) else torch.zeros_like(p)

    for i in range(la + 1):
        if i:
            v = e[(i - 1, 0)]
            e[(i, 0)] = [h * at(v, t - 1) + xpa * at(v, t) + (t + 1) * at(v, t + 1) for t in range(i + 1)]
        for j in range(1, lb + extra + 1):
            v = e[(i, j - 1)]
            e[(i, j)] = [h * at(v, t - 1) + xpb * at(v, t) + (t + 1) * at(v, t + 1) for t in range(i + j + 1)]
    return e


class _PairClass:
    """All primitive pairs of shells with l = (la, lb): centres, exponents, E[pair, ab component, Hermite]."""

    def __init__(self, sh, la, lb, cut=1e-18):
        pr = sh.prims()
        A, B = pr[la], pr[lb]
        fa, fb = (np.array([x[0] for x in s]) for s in (A, B))
        dev = sh.device
        xyz = sh.xyz.detach().cpu().numpy()
        ca, cb = (xyz[[x[1] for x in s]] for s in (A, B))
        ea, eb = (np.array([x[2] for x in s]) for s in (A, B))
        r2 = ((ca[:, None] - cb[None]) ** 2).sum(-1)
        k = np.exp(-ea[:, None] * eb[None] / (ea[:, None] + eb[None]) * r2)
        keep = k > cut
        if la == lb:
            keep &= fa[:, None] >= fb[None]
        ia, ib = np.nonzero(keep)
        self.count, self.la, self.lb = len(ia), la, lb

        def dev_of(v):
            return torch.as_tensor(np.ascontiguousarray(v), device=dev)

        self.fa, self.fb = dev_of(fa[ia]), dev_of(fb[ib])
        a, b = dev_of(ea[ia]), dev_of(eb[ib])
        RA = sh.xyz[dev_of(np.array([x[1] for x in A])[ia])]
        RB = sh.xyz[dev_of(np.array([x[1] for x in B])[ib])]
        c = dev_of((np.array([x[3] for x in A])[:, None] * np.array([x[3] for x in B])[None])[ia, ib])
        self.p = a + b
        self.P = (a[:, None] * RA + b[:, None] * RB) / self.p[:, None]
        d = RA - RB
        c = c * torch.exp(-a * b / self.p * (d * d).sum(1))
        self.c, self.b = c, b
        ax = [_expansion(la, lb, a, b, d[:, k], extra=2) for k in range(3)]
        self.ax = ax
        self.E = torch.stack([torch.stack([c * ax[0][(i[0], j[0])][h[0]] * ax[1][(i[1], j[1])][h[1]] *
                                           ax[2][(i[2], j[2])][h[2]]
                                           if all(h[k] <= i[k] + j[k] for k in range(3)) else torch.zeros_like(c)
                                           for h in _hermites(la + lb)], -1)
                              for i in _powers(la) for j in _powers(lb)], 1)

    def slots(self, index):
        """Rows index(fa + i, fb + j) of every pair's component block."""
        na, nb = len(_powers(self.la)), len(_powers(self.lb))
        dev = self.fa.device
        i = self.fa[:, None, None] + torch.arange(na, device=dev)[None, :, None]
        j = self.fb[:, None, None] + torch.arange(nb, device=dev)[None, None, :]
        return index(i, j).reshape(self.count, -1)


def _hermite_coulomb(l, alpha, X):
    """R_h for all h of total order <= l: dict of tensors shaped like alpha; X the three components."""
    t = alpha * (X[0] * X[0] + X[1] * X[1] + X[2] * X[2])
    f = _Boys.apply(t, l)
    base = []
    scale = torch.ones_like(alpha)
    for n in range(l + 1):
        base.append(scale * f[n])
        scale = scale * (-2.0 * alpha)
    level = {(0, 0, 0): base}  # h -> list over n
    for d in range(1, l + 1):
        for h in _powers(d):
            k = next(i for i in range(3) if h[i])
            lo = tuple(v - (i == k) for i, v in enumerate(h))
            lo2 = tuple(v - 2 * (i == k) for i, v in enumerate(h))
            out = []
            for n in range(l - d + 1):
                v = X[k] * level[lo][n + 1]
                if lo2[k] >= 0:
                    v = v + (h[k] - 1) * level[lo2][n + 1]
                out.append(v)
            level[h] = out
    return {h: v[0] for h, v in level.items()}


def _coulomb_block(bra, ket, lbra, lket, rows):
    """[pairs of bra in rows, ab, Q components] summed as Hermite interaction of two classes (ket: p, P, E)."""
    p, P, E = bra.p[rows], bra.P[rows], bra.E[rows]
    q, Qc, F = ket.p, ket.P, ket.E
    alpha = p[:, None] * q[None] / (p[:, None] + q[None])
    X = [P[:, None, k] - Qc[None, :, k] for k in range(3)]
    R = _hermite_coulomb(lbra + lket, alpha, X)
    pre = 2.0 * math.pi ** 2.5 / (p[:, None] * q[None] * torch.sqrt(p[:, None] + q[None]))
    hb, hk = _hermites(lbra), _hermites(lket)
    nb, nk, B, K = len(hb), len(hk), len(p), len(q)
    W = torch.stack([torch.stack([(-1.0 if sum(g) % 2 else 1.0) * R[tuple(x + y for x, y in zip(h, g))] for g in hk], -1)
                     for h in hb], 1)  # [bra, hb, ket, hk]
    W = W * pre[:, None, :, None]
    W = torch.bmm(E, W.reshape(B, nb, K * nk))  # [bra, ab, ket hk]
    W = W.reshape(B * E.shape[1], K, nk).transpose(0, 1).contiguous()
    W = torch.bmm(W, F.transpose(1, 2).contiguous())  # [ket, bra ab, cd]
    return W.reshape(K, B, E.shape[1], F.shape[1]).transpose(0, 1)  # [bra, ket, ab, cd]


def _classes(sh, cut=1e-18):
    ls = sorted(sh.prims())
    out = [_PairClass(sh, la, lb, cut) for la in ls for lb in ls if la >= lb]
    return [c for c in out if c.count]


def _chunks(count, size):
    for s in range(0, count, size):
        yield torch.arange(s, min(count, s + size))


def _one_electron(sh, classes, charges):
    n = sh.n
    S = torch.zeros(n * n, dtype=torch.float64, device=sh.device)
    T, V = S.clone(), S.clone()

    for c in classes:
        ax, b = c.ax, c.b
        s3 = (math.pi / c.p) ** 1.5 * c.c

        def ov(k, i, j):
            return ax[k][(i, j)][0] if j >= 0 else torch.zeros_like(b)

        def kin(k, i, j):
            v = -2.0 * b * b * ov(k, i, j + 2) + b * (2 * j + 1) * ov(k, i, j)
            return v - 0.5 * j * (j - 1) * ov(k, i, j - 2) if j >= 2 else v

        sb, tb = [], []
        for i in _powers(c.la):
            for j in _powers(c.lb):
                o = [ov(k, i[k], j[k]) for k in range(3)]
                t = [kin(k, i[k], j[k]) for k in range(3)]
                sb.append(s3 * o[0] * o[1] * o[2])
                tb.append(s3 * (t[0] * o[1] * o[2] + o[0] * t[1] * o[2] + o[0] * o[1] * t[2]))
        L = c.la + c.lb
        alpha = c.p[:, None].expand(-1, len(charges))
        R = _hermite_coulomb(L, alpha, [c.P[:, None, k] - sh.xyz[None, :, k] for k in range(3)])
        pot = torch.stack([-(R[h] * charges[None]).sum(1) for h in _hermites(L)], -1)
        vb = torch.matmul(c.E, pot[..., None])[..., 0] * (2.0 * math.pi / c.p)[:, None]
        at = c.slots(lambda i, j: i * n + j).reshape(-1)
        S = S.index_add(0, at, torch.stack(sb, 1).reshape(-1))
        T = T.index_add(0, at, torch.stack(tb, 1).reshape(-1))
        V = V.index_add(0, at, vb.reshape(-1))
    out = []
    fac, slot = sh.factors()
    for m in (S, T, V):
        m = m.reshape(n, n)
        low = _from_blocks(sh, m)
        out.append(low[slot][:, slot] * fac[:, None] * fac[None])
    return out


def _shell_of(sh):
    first = np.zeros(sh.n, np.int64)
    for l, _, f, _, _, _, _ in sh.rows:
        first[f:f + (l + 1) * (l + 2) // 2] = f
    lof = np.zeros(sh.n, np.int64)
    for l, _, f, _, _, _, _ in sh.rows:
        lof[f:f + (l + 1) * (l + 2) // 2] = l
    return torch.as_tensor(first, device=sh.device), torch.as_tensor(lof, device=sh.device)


def _from_blocks(sh, m):
    """A symmetric matrix from its blocks held once, at (higher l, or the later shell of equal l)."""
    first, l = _shell_of(sh)
    held = (l[:, None] > l[None]) | ((l[:, None] == l[None]) & (first[:, None] >= first[None]))
    return torch.where(held, m, m.transpose(0, 1))


def _eri(sh, classes):
    """(ij|kl) as [n*n, n*n] over the ordered blocks, then symmetrised on both sides."""
    n = sh.n
    G = torch.zeros((n * n) * (n * n), dtype=torch.float64, device=sh.device)
    for c in classes:
        ra = c.slots(lambda i, j: i * n + j)
        for d in classes:
            rd = d.slots(lambda i, j: i * n + j)
            size = max(1, int(2e7 / (d.count * max(c.E.shape[2] * d.E.shape[2], c.E.shape[1] * d.E.shape[1]))))
            for rows in _chunks(c.count, size):
                blk = _coulomb_block(c, d, c.la + c.lb, d.la + d.lb, rows.to(sh.device))
                at = ra[rows.to(sh.device)][:, None, :, None] * (n * n) + rd[None, :, None, :]
                G = G.index_add(0, at.reshape(-1), blk.reshape(-1))
    fac, slot = sh.factors()
    first, l = _shell_of(sh)
    held = (l[:, None] > l[None]) | ((l[:, None] == l[None]) & (first[:, None] >= first[None]))
    ij = torch.arange(n * n, device=sh.device).reshape(n, n)
    src = torch.where(held, ij, ij.transpose(0, 1))[slot][:, slot].reshape(-1)
    ff = (fac[:, None] * fac[None]).reshape(-1)
    G = G.reshape(n * n, n * n)[src][:, src]
    return G * ff[:, None] * ff[None]


def _jk_of(G, P):
    n = P.shape[0]
    J = (G @ P.reshape(-1)).reshape(n, n)
    K = torch.einsum("ikjl,kl->ij", G.reshape(n, n, n, n), P)
    return J, K


class _AuxClass:
    """The shells of one l of an auxiliary basis as Hermite charges."""

    def __init__(self, sh, l):
        pr = sh.prims()[l]
        dev = sh.device
        self.f = torch.as_tensor(np.array([x[0] for x in pr]), device=dev)
        a = torch.as_tensor(np.array([x[2] for x in pr]), device=dev)
        c = torch.as_tensor(np.array([x[3] for x in pr]), device=dev)
        self.p, self.P, self.count, self.l = a, sh.xyz[torch.as_tensor(np.array([x[1] for x in pr]), device=dev)], len(pr), l
        ax = _expansion(l, 0, a, torch.zeros_like(a), torch.zeros_like(a))
        self.E = torch.stack([torch.stack([c * ax[(i[0], 0)][h[0]] * ax[(i[1], 0)][h[1]] * ax[(i[2], 0)][h[2]]
                                           if all(h[k] <= i[k] for k in range(3)) else torch.zeros_like(c)
                                           for h in _hermites(l)], -1) for i in _powers(l)], 1)

    def slots(self):
        return self.f[:, None] + torch.arange(len(_powers(self.l)), device=self.f.device)[None]


def _df_jk(basis, auxb, xyz, C, cutoff, device):
    """J and K of the fitted integrals: metric, its orthogonaliser above the cutoff, (P|mn), and the contractions."""
    sh, au = _Shells(basis, xyz, device), _Shells(auxb, xyz, device)
    n, na, o = sh.n, au.n, C.shape[1]
    facs, slots = sh.factors()
    faca, slota = au.factors()
    ac = [_AuxClass(au, l) for l in sorted(au.prims())]
    V = torch.zeros((na, na), dtype=torch.float64, device=device)
    for c in ac:
        for d in ac:
            blk = _coulomb_block(c, d, c.l, d.l, torch.arange(c.count, device=device))
            at = c.slots()[:, None, :, None] * na + d.slots()[None, :, None, :]
            V.view(-1).index_add_(0, at.reshape(-1), blk.reshape(-1))
    V = V[slota][:, slota] * faca[:, None] * faca[None]
    w, U = torch.linalg.eigh(V)
    X = (U / torch.sqrt(w.clamp_min(1e-300)))[:, w >= cutoff]
    T = torch.zeros(na * n * n, dtype=torch.float64, device=device)
    for c in _classes(sh):
        ra = c.slots(lambda i, j: i * n + j)
        for d in ac:
            size = max(1, int(6e7 / (d.count * max(c.E.shape[2] * d.E.shape[2], c.E.shape[1] * d.E.shape[1]))))
            for rows in _chunks(c.count, size):
                rows = rows.to(device)
                blk = _coulomb_block(c, d, c.la + c.lb, d.l, rows)
                at = d.slots()[None, :, None, :] * (n * n) + ra[rows][:, None, :, None]
                T.index_add_(0, at.reshape(-1), blk.reshape(-1))
    T = T.reshape(na, n, n)
    for q in range(na):
        T[q] = _from_blocks(sh, T[q])[slots][:, slots] * facs[:, None] * facs[None]
    src = slota
    if not torch.equal(src, torch.arange(na, device=device)):
        T = T[src]
    T *= faca[:, None, None]
    P = 2.0 * C @ C.T
    d = X.T @ (T.reshape(na, -1) @ P.reshape(-1))
    J = ((X @ d) @ T.reshape(na, -1)).reshape(n, n)
    A = X.T @ torch.matmul(T, C).reshape(na, n * o)
    del T
    A = A.reshape(-1, n, o).transpose(0, 1).reshape(n, -1)
    return J, 2.0 * A @ A.T


def _gradient(state, device):
    xyz = torch.tensor(state["mol"].xyz, dtype=torch.float64, device=device, requires_grad=True)
    sh = _Shells(state["basis"], xyz, device)
    z = torch.as_tensor(state["mol"].zxyz[:, 0].copy(), device=device)
    P, W = (torch.as_tensor(state[k], device=device) for k in ("p", "w"))
    cl = _classes(sh)
    S, T, V = _one_electron(sh, cl, z)
    J, K = _jk_of(_eri(sh, cl), P)
    e = (P * (T + V)).sum() + 0.5 * (P * J).sum() - 0.25 * (P * K).sum() - (W * S).sum()
    i, j = torch.triu_indices(len(z), len(z), 1, device=device)
    e = e + (z[i] * z[j] / (xyz[i] - xyz[j]).norm(dim=1)).sum()
    e.backward()
    return xyz.grad


def _rhf(state, device):
    """RHF to convergence: commutator DIIS from the core Hamiltonian."""
    xyz = torch.as_tensor(state["mol"].xyz, device=device)
    z = torch.as_tensor(state["mol"].zxyz[:, 0].copy(), device=device)
    sh = _Shells(state["basis"], xyz, device)
    cl = _classes(sh)
    S, T, V = _one_electron(sh, cl, z)
    G = _eri(sh, cl)
    o = state["mol"].n_electrons() // 2
    w, U = torch.linalg.eigh(S)
    X = (U / torch.sqrt(w))[:, w >= 1e-8]
    H = T + V
    i, j = torch.triu_indices(len(z), len(z), 1, device=device)
    enuc = (z[i] * z[j] / (xyz[i] - xyz[j]).norm(dim=1)).sum()

    def density(F):
        c = X @ torch.linalg.eigh(X.T @ F @ X)[1][:, :o]
        return 2.0 * c @ c.T

    P, hist = density(H), []
    for _ in range(150):
        J, K = _jk_of(G, P)
        F = H + J - 0.5 * K
        err = X.T @ (F @ P @ S - S @ P @ F) @ X
        hist = (hist + [(F, err)])[-8:]
        if float(err.abs().max()) < 1e-11:
            break
        k = len(hist)
        B = torch.full((k + 1, k + 1), -1.0, dtype=torch.float64, device=device)
        B[k, k] = 0.0
        for a in range(k):
            for b in range(k):
                B[a, b] = (hist[a][1] * hist[b][1]).sum()
        B[:k, :k] /= B[:k, :k].abs().max()
        rhs = torch.zeros(k + 1, 1, dtype=torch.float64, device=device)
        rhs[k] = -1.0
        c = torch.linalg.lstsq(B.cpu(), rhs.cpu(), driver="gelsd").solution[:k, 0].to(device)
        P = density(sum(c[a] * hist[a][0] for a in range(k)))
    else:
        return None
    return {"energy": float(0.5 * ((P * H).sum() + (P * F).sum()) + enuc), "density": P, "fock": F}


def exact(case, seed):
    path = case["path"]
    rng = _rng(case, seed)
    if path in ("batch", "server", "df_rhf"):
        return None
    mol = _molecule(case, rng)
    basis = _basis(case["basis"], mol)
    n, o = basis.n, mol.n_electrons() // 2
    device = "cuda" if torch.cuda.is_available() else "cpu"
    state = {"mol": mol, "basis": basis}
    xyz = torch.as_tensor(mol.xyz, device=device)
    if path == "df":
        aux = _basis(AUX[case["basis"]], mol)
        c = torch.as_tensor(_orbitals(n, o, rng), device=device)
        if float(aux.n) * n * n > 3.5e9:
            return None
        return _df_jk(basis, aux, xyz, c, 1e-10, device)
    if n > {"jk": 110, "scf": 90, "grad": 26}[path]:
        return None
    if path == "scf":
        return _rhf(state, device)
    c = _orbitals(n, o, rng)
    state["p"] = 2.0 * c @ c.T
    if path == "grad":
        eps = -np.sort(rng.uniform(0.3, 20.0, o))[::-1]
        state["w"] = 2.0 * (c * eps) @ c.T
        return _gradient(state, device)
    sh = _Shells(basis, xyz, device)
    return _jk_of(_eri(sh, _classes(sh)), torch.as_tensor(state["p"], device=device))
