"""Performance cases of the magnetic-ACE evaluator: the work that its users have it do, through
the entry points they call, over the sizes they use.

A case is a dict of plain values; its ``kind`` says which program it stands for:

* ``eval``  a GPU-resident driver: pair arrays on the device, one energy / force / torque
            evaluation (``capi.compute_device``).  In mixed precision such a driver keeps its
            results as float32, the precision the arithmetic has; in FP64 it keeps them as
            they come.
* ``host``  LAMMPS pair_spin_ace: the same evaluation through ``acelib_`` on host arrays, in the
            precision LAMMPS gets without asking (FP64).
* ``neigh`` a neighbour-list rebuild on the device (one system, or a batch of structures).
* ``fit``   one training step: energies and forces of a batch of structures, a quadratic loss,
            the gradient in the expansion coefficients.
* ``md``    ten steps of spin-lattice dynamics (one list rebuild, the graph-replayed steps) and
            the frame read back, which a trajectory keeps as float32.

``listed()`` are the cases that are measured, ``draw(rng)`` gives others of the same ranges,
``exact(case, seed)`` evaluates the potential in 64 bits with torch alone, from the text of the
potential file.
"""
import math
import os
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

import __graft_entry__  # noqa: E402

PKG = __graft_entry__.load_package()
capi = PKG.capi

#: potential headers by name: lmax 4 with 489 B functions and lmax 6 with 2043 (the two that the
#: benchmark and the tests evaluate), the shape of the example potential (27 magnetic columns,
#: nonlinear embedding), the lmax-4 header with two densities
HEADERS = {"lmax4": PKG.potgen.H500, "lmax6": PKG.potgen.H2000, "wide": PKG.potgen.HFE,
           "twodens": PKG.potgen.H500ND2}
RCUT, RCUT_M = 5.0, 4.0
#: pairs an atom that a program leaves room for: bcc Fe has 58 neighbours within 5 A, and the next shell
#: is 0.66 A further out
MOST = 60


def listed():
    return [
        # one spin's surroundings, as a spin sweep or an energy difference of a small cell asks for
        # it: a call of a hundred-odd microseconds, where launches and host work are what counts
        dict(name="host fp64 lmax4 54", kind="host", header="lmax4", n1=3, n2=3, n3=3, vac=0, spins="uniform"),
        # the 128-atom cell with non-collinear spins: relaxations, convergence tests
        dict(name="eval fp64 lmax4 128", kind="eval", header="lmax4", precision="fp64", n1=4, n2=4, n3=4, vac=0, spins="uniform"),
        # a supercell with a vacancy, FP64: defect energies
        dict(name="eval fp64 lmax6 431", kind="eval", header="lmax6", precision="fp64", n1=6, n2=6, n3=6, vac=1, spins="cone"),
        # the 2000-atom cell in mixed precision: ordinary dynamics of one cell
        dict(name="eval mixed lmax4 2000", kind="eval", header="lmax4", precision="mixed", n1=10, n2=10, n3=10, vac=0, spins="uniform"),
        # the example potential's shape, mixed, a box with unequal edges and two vacancies
        dict(name="eval mixed wide 4366", kind="eval", header="wide", precision="mixed", n1=12, n2=13, n3=14, vac=2, spins="uniform"),
        # the same potential shape in FP64, an ordinary cell
        dict(name="eval fp64 wide 1024", kind="eval", header="wide", precision="fp64", n1=8, n2=8, n3=8, vac=0, spins="uniform"),
        # the 16000-atom headline workload, in both precisions
        dict(name="eval mixed lmax6 16000", kind="eval", header="lmax6", precision="mixed", n1=20, n2=20, n3=20, vac=0, spins="cone"),
        dict(name="eval fp64 lmax6 16000", kind="eval", header="lmax6", precision="fp64", n1=20, n2=20, n3=20, vac=0, spins="cone"),
        # the same call as LAMMPS makes it: host arrays, copies included
        dict(name="host fp64 lmax6 6750", kind="host", header="lmax6", n1=15, n2=15, n3=15, vac=0, spins="cone"),
        # the list rebuild that every driver runs each few steps
        dict(name="neigh 16000", kind="neigh", header="lmax4", confs=1, n1=20, n2=20, n3=20, vac=0, spins="uniform"),
        # one step of a fit over 256 structures of 16 to 1024 atoms
        dict(name="fit lmax4 256", kind="fit", header="lmax4", confs=256, lo=16, hi=1024),
        # the large dynamics run: 128000 atoms
        dict(name="md mixed lmax4 128000", kind="md", header="lmax4", precision="mixed", n1=40, n2=40, n3=40, vac=0, spins="uniform"),
    ]


def _box(rng, lo, hi):
    """Cells along three edges, the number of atoms spread over lo..hi on its logarithm."""
    cells = math.exp(rng.uniform(math.log(lo), math.log(hi))) / 2
    a = cells ** (1 / 3)
    n1 = max(1, round(a * rng.uniform(0.75, 1.25)))
    n2 = max(1, round(math.sqrt(cells / n1) * rng.uniform(0.85, 1.15)))
    return dict(n1=n1, n2=n2, n3=max(1, round(cells / (n1 * n2))))


def draw(rng):
    kind = rng.choice(["eval"] * 6 + ["host", "neigh", "fit", "md"])
    spins = rng.choice(["uniform", "cone"])
    header = rng.choice(["lmax4", "lmax6", "wide", "twodens"])
    precision = rng.choice(["fp64", "mixed"])
    vac = rng.randint(0, 2)
    if kind == "eval":
        return dict(kind=kind, header=header, precision=precision, **_box(rng, 24, 16000), vac=vac, spins=spins)
    if kind == "host":
        return dict(kind=kind, header=header, **_box(rng, 24, 8000), vac=vac, spins=spins)
    if kind == "neigh":
        if rng.random() < 0.5:
            lo = rng.randint(16, 64)
            return dict(kind=kind, header="lmax4", confs=rng.randint(4, 128), lo=lo, hi=lo * rng.randint(2, 8))
        return dict(kind=kind, header="lmax4", confs=1, **_box(rng, 100, 50000), vac=vac, spins=spins)
    if kind == "fit":
        lo = rng.randint(16, 64)
        return dict(kind=kind, header=rng.choice(["lmax4", "lmax4", "lmax6"]), confs=rng.randint(4, 96), lo=lo,
                    hi=lo * rng.randint(2, 8))
    return dict(kind=kind, header="lmax4", precision=precision, **_box(rng, 250, 32000), vac=vac, spins=spins)


# ---------------------------------------------------------------- inputs

_loaded = None  # (header, whether a fit set its coefficients) of the potential in the library


def _text(header):
    h = HEADERS[header]
    return PKG.potgen.render(h, capi.enumerate_basis(h), 2026)


def _load(header, fit=False):
    """The potential in the library (a program loads its potential once)."""
    global _loaded
    if _loaded != (header, fit):
        with tempfile.TemporaryDirectory() as d:
            path = os.path.join(d, "Fe.pbe.in")
            with open(path, "w") as f:
                f.write(_text(header))
            capi.init_file(path, rcut=RCUT, rcut_magnetic=RCUT_M)
        _loaded = (header, fit)


def _system(case, seed):
    """bcc Fe, jittered by N(0, 0.05 A), with `vac` atoms taken out; moments N(2.2, 0.1) muB,
    directions uniform on the sphere or in a cone of 30 degrees about z."""
    rng = np.random.default_rng(seed)
    pos, cell = PKG.systems.bcc_box(case["n1"], case["n2"], case["n3"])
    if case["vac"] and len(pos) > case["vac"] + 1:
        pos = np.delete(pos, rng.choice(len(pos), case["vac"], replace=False), axis=0)
    pos = PKG.systems.jitter(pos, rng, 0.05)
    spins = PKG.systems.spins_cone if case["spins"] == "cone" else PKG.systems.spins_uniform
    sdir, smag = spins(len(pos), rng)
    return dict(pos=pos, cell=cell, sdir=sdir, smag=smag, rng=rng)


def _structures(case, seed):
    """One system, or `confs` periodic bcc structures of lo..hi atoms (spread over the logarithm; the
    sizes and the 0-2 vacancies belong to the case), strained by up to 3%, jittered, spins at random."""
    if case.get("confs", 1) == 1:
        return [_system(case, seed)]
    sizes, rng, out = np.random.default_rng(2029), np.random.default_rng(seed), []
    for _ in range(case["confs"]):
        cells = max(1.0, math.exp(sizes.uniform(math.log(case["lo"]), math.log(case["hi"]))) / 2)
        n1 = max(1, round(cells ** (1 / 3)))
        n2 = max(1, round(math.sqrt(cells / n1)))
        pos, cell = PKG.systems.bcc_box(n1, n2, max(1, round(cells / (n1 * n2))), PKG.systems.A_FE * (1 + rng.uniform(-0.03, 0.03)))
        vac = int(sizes.integers(0, 3))
        if len(pos) > vac + 1:
            pos = np.delete(pos, rng.choice(len(pos), vac, replace=False), axis=0)
        sdir, smag = PKG.systems.spins_uniform(len(pos), rng)
        out.append(dict(pos=PKG.systems.jitter(pos, rng, 0.05), cell=cell, sdir=sdir, smag=smag))
    return out


def _lists(structures):
    """Device neighbour lists of the structures, packed one after another, in arrays that hold MOST
    pairs an atom."""
    natoms = np.array([len(s["pos"]) for s in structures], np.int32)
    nb = PKG.neighbors.DeviceNeighbors(natoms, [1] * len(structures), np.stack([s["cell"] for s in structures]), RCUT,
                                       capacity=MOST * int(natoms.sum()))
    pos = torch.tensor(np.concatenate([s["pos"] for s in structures]), device="cuda")
    mag = torch.tensor(np.concatenate([s["sdir"] * s["smag"][:, None] for s in structures]), device="cuda")
    return nb, pos, mag


def prepare(case, seed):
    kind = case["kind"]
    if kind == "neigh":
        nb, pos, mag = _lists(_structures(case, seed))
        return dict(kind=kind, nb=nb, pos=pos, mag=mag)
    if kind == "fit":
        _load(case["header"], True)
        structures = _structures(case, seed)
        batch = PKG.fit.Batch(structures, RCUT)
        rng = np.random.default_rng([seed, 1])
        n = torch.tensor(batch.natoms, dtype=torch.float64, device="cuda")
        return dict(kind=kind, batch=batch, weight=1.0 / n,
                    c=torch.tensor(rng.normal(0.0, 1e-2, capi.fit_ncoef()), device="cuda", requires_grad=True),
                    E0=torch.tensor(rng.normal(0.0, 0.2, batch.nstruc), device="cuda") * n,
                    F0=torch.tensor(rng.normal(0.0, 0.3, (batch.natom, 3)), device="cuda"))
    _load(case["header"])
    capi.set_precision(capi.MIXED if case.get("precision") == "mixed" else capi.FP64)
    s = _system(case, seed)
    if kind == "md":
        vel = PKG.md.maxwell_velocities(len(s["pos"]), 300.0, s["rng"])
        return dict(kind=kind, md=PKG.md.SpinLatticeMD(s["pos"], s["cell"], s["sdir"], s["smag"], vel, dt=1e-4, rcut=RCUT))
    nb, pos, mag = _lists([s])
    L = {k: v.clone() for k, v in nb.build(pos, mag).items() if k != "npairs"}
    N, P = len(s["pos"]), len(L["dlist"])
    if kind == "host":
        a = {k: v.cpu().numpy() for k, v in L.items()}
        off = a["offsets"]
        a = dict(natom=N, nall=N, nstart=off[:-1] + np.int32(1), nstop=off[1:].copy(), nlist=a["nlist"] + np.int32(1),
                 occ=np.ones(N, np.int32), occlist=np.ones(P, np.int32),
                 **{k: a[k] for k in ("dlist", "elist", "dlist_mom", "elist_mom", "dlist_momi", "elist_momi")})
        out = dict(eout=np.zeros(N), flist=np.zeros((MOST * N, 3)), tlist=np.zeros((MOST * N, 3)), tlist0=np.zeros((N, 3)))
        views = (out["eout"], out["flist"].reshape(-1)[:3 * P], out["tlist"].reshape(-1)[:3 * P], out["tlist0"].reshape(-1))
        return dict(kind=kind, a=a, L=L, out=out, views=dict(_buffers=views))  # the caller keeps its output arrays
    out = dict(eout=torch.zeros(N, dtype=torch.float64, device="cuda"),
               flist=torch.zeros(MOST * N, 3, dtype=torch.float64, device="cuda"),
               tlist=torch.zeros(MOST * N, 3, dtype=torch.float64, device="cuda"),
               tlist0=torch.zeros(N, 3, dtype=torch.float64, device="cuda"))
    kept = {k: torch.zeros_like(v, dtype=torch.float32) for k, v in out.items()} if case["precision"] == "mixed" else None
    return dict(kind=kind, L=L, N=N, P=P, out=out, kept=kept)


# ---------------------------------------------------------------- one pass

def run(state):
    kind = state["kind"]
    if kind == "eval":
        L, o = state["L"], state["out"]
        capi.compute_device(state["N"], state["P"], L["offsets"].data_ptr(), L["dlist"].data_ptr(), L["elist"].data_ptr(),
                            L["dlist_momi"].data_ptr(), L["elist_momi"].data_ptr(), L["dlist_mom"].data_ptr(),
                            L["elist_mom"].data_ptr(), o["eout"].data_ptr(), o["flist"].data_ptr(),
                            o["tlist"].data_ptr(), o["tlist0"].data_ptr(), torch.cuda.current_stream().cuda_stream)
        if state["kept"] is None:
            return o
        for k, v in state["kept"].items():
            v.copy_(o[k])
        return state["kept"]
    if kind == "host":
        capi.acelib(state["a"], state["views"])
        return state["out"]
    if kind == "neigh":
        nb = state["nb"]
        r = nb.build(state["pos"], state["mag"])
        return dict(npairs=r["npairs"], offsets=nb.offsets, nlist=nb.nlist, dlist=nb.dlist, elist=nb.elist,
                    dlist_mom=nb.dlist_mom, elist_mom=nb.elist_mom, dlist_momi=nb.dlist_momi, elist_momi=nb.elist_momi)
    if kind == "fit":
        c = state["c"]
        c.grad = None
        E, F = PKG.fit.EnergyForces.apply(c, state["batch"])
        loss = (state["weight"] * (E - state["E0"])).square().sum() + (F - state["F0"]).square().sum()
        loss.backward()
        return dict(E=E.detach(), F=F.detach(), grad=c.grad)
    md = state["md"]
    md.run(10)
    st = md.state()
    frame = {k: st[k].astype(np.float32) for k in ("x", "v", "sdir", "f", "dEdm", "eatom")}
    return dict(frame, epot=np.float32(st["epot"]), ekin=np.float32(st["ekin"]))


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    """Bytes: each input read once, each output written once.  Flops: the density accumulation
    over the pairs and its derivative contracted with dE/dA (half of each by conjugate symmetry),
    the radial functions and harmonics of each pair, and the monomials of the basis with their
    gradient."""
    h = HEADERS[case["header"]]
    kind = case["kind"]
    if case.get("confs", 1) > 1:
        N = case["confs"] * (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
    else:
        N = 2 * case["n1"] * case["n2"] * case["n3"] - case["vac"]
    P = 57.5 * N
    if kind == "neigh":
        return dict(bytes=48 * N + 36 * N + 68 * P, flops=40 * P)
    lha, lhm = (h["l3a"] + 1) * (h["l3a"] + 2) / 2, (h["l2m"] + 1) * (h["l2m"] + 2) / 2
    nA = h["nr3_a"] * lha * h["nr3_m"] * (h["l3m"] + 1) ** 2
    nA2 = h["nb_a"] * h["nr2_m"] * lhm
    radial = h["nb_a"] + h["nr3_a"] * (h["l3a"] + 1) + h["nb_m"] + h["nr2_m"] * (h["l2m"] + 1)
    pair = 11 * radial + 30 * (lha + lhm) + 4 * (nA + nA2) + 8 * (nA + nA2)
    terms = {"lmax4": 3636, "lmax6": 31272, "wide": 35757, "twodens": 2 * 3636}[case["header"]]
    flops = P * pair + N * 16.0 * terms
    steps = 10 if kind == "md" else 1
    passes = 2 if kind == "fit" else 1  # a fit's gradient runs through the density and the monomials again
    move = 112 * P + 64 * N if kind in ("eval", "host") else 48 * P + 100 * N
    return dict(bytes=float(steps * move), flops=float(steps * passes * flops))


# ---------------------------------------------------------------- the same in 64 bits, with torch alone

class _Exact:
    """The potential of a text file, evaluated with torch in 64 bits from its definition: spline
    radial functions, A = sum_j R Y (M Y'), coupled products, embedding; gradients by autograd."""

    def __init__(self, text):
        L = text.split("\n")
        num = lambda i: [float(t) for t in L[i].replace("rcut dcut ecut decut", "").split() if t[0] in "-0123456789."]  # noqa: E731
        self.lam, self.cut = num(5), num(6)
        self.nba, self.nbm, self.nr2m, self.l2m = (int(t) for t in L[7].split()[-4:])
        self.nr3a, self.nr3m, self.l3a, self.l3m = (int(t) for t in L[8].split()[-4:])
        self.nd = int(L[12].split()[-1])
        _, self.nfemb, ta, tm = (int(t) for t in L[13].split()[-4:])
        assert (ta, tm) == (3, 7)
        self.ca = np.zeros((self.nr3a, self.l3a + 1, self.nba))
        self.cm = np.zeros((self.nr2m, self.l2m + 1, self.nbm))
        self.par, self.core = {}, {}
        self.clu = {}  # (order, density) -> list of (indices, coefficient)
        for head, rec in zip(L[14::2], L[15::2]):
            a, b, d = head.split()[0], int(head.split()[1]), int(head.split()[2])
            t = [v for v in rec.split() if v not in ("Fe", "T", "F")]
            if a == "par":
                self.par[b, d] = float(t[0])
            elif a == "core":
                self.core[b] = float(t[0])
            elif a == "rad_atomic":
                self.ca[int(t[1]) - 1, int(t[2]), int(t[0]) - 1] = float(t[3])
            elif a == "rad_magnetic":
                self.cm[int(t[1]) - 1, int(t[2]), int(t[0]) - 1] = float(t[3])
            elif a == "clu":
                self.clu.setdefault((b, d), []).append(([int(v) for v in t[:-1]], float(t[-1])))
        assert self.core[1] == 0.0
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self._tables()
        self._terms()

    def _tables(self):
        """Cubic Hermite tables of the radial functions at x_n = n rc / 10000, n = 1..10000."""
        nlut = self.nlut = 10000
        cheb = np.polynomial.chebyshev

        def hermite(f, df, step):  # [nlut, nf]
            d = df * step
            f1, d1 = np.vstack([f[1:], 0 * f[:1]]), np.vstack([d[1:], 0 * d[:1]])
            c = np.stack([f, d, 3 * (f1 - f) - d1 - 2 * d, -2 * (f1 - f) + d1 + d], axis=2)
            return torch.tensor(c, device=self.dev)

        def smooth(g, dg, r, cut, dcut):
            lo = cut - dcut
            on = r > lo
            fc = np.where(on, 0.5 * (1 + np.cos(np.pi * (r - lo) / dcut)), 1.0)[:, None]
            dfc = np.where(on, -0.5 * np.sin(np.pi * (r - lo) / dcut) * np.pi / dcut, 0.0)[:, None]
            out = (r >= cut)[:, None]
            return np.where(out, 0.0, g * fc), np.where(out, 0.0, g * dfc + dg * fc)

        def chebyshev(n, x):
            t = np.stack([cheb.chebval(x, np.eye(n + 1)[k]) for k in range(n + 1)], 1)
            dt = np.stack([cheb.chebval(x, cheb.chebder(np.eye(n + 1)[k])) if k else 0 * x for k in range(n + 1)], 1)
            return t, dt

        r, cut, lam = RCUT / nlut * np.arange(1, nlut + 1), self.cut[0], self.lam[0]
        y1, y2 = np.exp(-lam * r / cut), math.exp(-lam)
        t, dt = chebyshev(self.nba - 1, 1 - 2 * (y1 - y2) / (1 - y2))
        dx = (2 * lam * y1 / (cut * (1 - y2)))[:, None]
        g, dg = 0.5 - 0.5 * t, -0.5 * dt * dx
        g[:, 0], dg[:, 0] = 1.0, 0.0
        env, denv = 0.5 * (1 + np.cos(np.pi * r / cut))[:, None], (-0.5 * np.sin(np.pi * r / cut) * np.pi / cut)[:, None]
        g, dg = smooth(g * env, g * denv + dg * env, r, cut, self.cut[2])
        R, dR = (np.einsum("nlk,xk->xln", self.ca, v).reshape(nlut, -1) for v in (g, dg))
        self.tab_a = hermite(np.hstack([g, R]), np.hstack([dg, dR]), RCUT / nlut)

        r, cut = RCUT_M / nlut * np.arange(1, nlut + 1), self.cut[1]
        t, dt = chebyshev(self.nbm, 1 - 2 * (r / cut) ** 2)
        g, dg = smooth(t[:, 1:], dt[:, 1:] * (-4 * r / cut ** 2)[:, None], r, cut, self.cut[3])
        M, dM = (np.einsum("nlk,xk->xln", self.cm, v).reshape(nlut, -1) for v in (g, dg))
        self.tab_m = hermite(np.hstack([g, M]), np.hstack([dg, dM]), RCUT_M / nlut)

    def _spline(self, tab, r, cut):
        x = r * (self.nlut / cut)
        n = torch.floor(x.detach())
        w = (x - n)[:, None]
        c = tab[(n.long() - 1).clamp(0, self.nlut - 1)]
        v = ((c[:, :, 3] * w + c[:, :, 2]) * w + c[:, :, 1]) * w + c[:, :, 0]
        return torch.where((n >= self.nlut)[:, None], torch.zeros_like(v), v)

    def _harmonics(self, u, lmax):
        """Y_lm of the unit vectors u, sqrt(4 pi) times the Condon-Shortley ones: [.., (l, m)], real and imaginary."""
        x, y, z = u.unbind(-1)
        pr, pi = [torch.ones_like(x)], [torch.zeros_like(x)]
        for _ in range(lmax):
            pr, pi = pr + [pr[-1] * x - pi[-1] * y], pi + [pr[-1] * y + pi[-1] * x]
        re, im = [], []
        for l in range(lmax + 1):
            row = {}
            for m in range(l + 1):
                p = np.polynomial.legendre.leg2poly(np.eye(l + 1)[l])
                for _ in range(m):
                    p = np.polynomial.polynomial.polyder(p)
                norm = (-1) ** m * math.sqrt((2 * l + 1) * math.factorial(l - m) / math.factorial(l + m))
                v = torch.zeros_like(z)
                for c in p[::-1]:
                    v = v * z + float(c) * norm
                row[m] = (v * pr[m], v * pi[m])
            for m in range(-l, l + 1):
                s = (-1) ** m if m < 0 else 1
                re.append(s * row[abs(m)][0])
                im.append(s * row[abs(m)][1] if m >= 0 else -s * row[abs(m)][1])
        return torch.stack(re, -1), torch.stack(im, -1)

    @staticmethod
    def _cg(j1, j2, J, m1, m2, M, memo={}):
        key = (j1, j2, J, m1, m2, M)
        if key in memo:
            return memo[key]
        f = math.factorial
        v = 0.0
        if m1 + m2 == M and abs(j1 - j2) <= J <= j1 + j2 and abs(M) <= J and abs(m1) <= j1 and abs(m2) <= j2:
            pre = math.sqrt((2 * J + 1) * f(J + j1 - j2) * f(J - j1 + j2) * f(j1 + j2 - J) / f(j1 + j2 + J + 1))
            pre *= math.sqrt(f(J + M) * f(J - M) * f(j1 - m1) * f(j1 + m1) * f(j2 - m2) * f(j2 + m2))
            for k in range(j1 + j2 + J + 1):
                d = (k, j1 + j2 - J - k, j1 - m1 - k, j2 + m2 - k, J - j2 + m1 + k, J - j1 - m2 + k)
                if min(d) >= 0:
                    v += (-1) ** k / math.prod(f(t) for t in d)
            v *= pre
        memo[key] = v
        return v

    def _terms(self):
        """Products of columns of Z = [A | A2 | A0 | 1] with their coupling, summed over equal products:
        rho_d = Re sum_t (sum_k c_kd U_kt) prod_s Z[idx_ts]."""
        lsa, lsm, ls3 = (self.l3a + 1) ** 2, (self.l2m + 1) ** 2, (self.l3m + 1) ** 2
        nq = self.nr3m * ls3
        oA2 = self.nr3a * lsa * nq
        oA0 = oA2 + self.nba * self.nr2m * lsm
        one = self.one = oA0 + self.nr2m * lsm
        A = lambda n, l, m, np_, lp, mp: ((n - 1) * lsa + l * l + l + m) * nq + (np_ - 1) * ls3 + lp * lp + lp + mp  # noqa: E731
        A2 = lambda n, np_, l, m: oA2 + ((n - 1) * self.nr2m + np_ - 1) * lsm + l * l + l + m  # noqa: E731
        A0 = lambda np_, l, m: oA0 + (np_ - 1) * lsm + l * l + l + m  # noqa: E731
        cg, idx, k_of, t_of, u_of = self._cg, {}, [], [], []

        def emit(k, u, *cols):
            if u:
                t = idx.setdefault(tuple(sorted(cols + (one,) * (4 - len(cols)))), len(idx))
                k_of.append(k), t_of.append(t), u_of.append(u)

        k = 0
        for b, _ in self.clu.get((2, 1), []):
            n0, n1p, n1, l = b
            for m in range(-l, l + 1):
                emit(k, cg(l, l, 0, m, -m, 0), A0(n0, l, m), A2(n1, n1p, l, -m))
            k += 1
        for b, _ in self.clu.get((3, 1), []):
            n1, n2, n0p, n1p, n2p, l, l0, l1, l2 = b
            for m in range(-l, l + 1):
                for q0 in range(-l0, l0 + 1):
                    for q1 in range(-l1, l1 + 1):
                        q2 = -q0 - q1
                        if abs(q2) <= l2:
                            u = cg(l, l, 0, m, -m, 0) * cg(l0, l1, l2, q0, q1, -q2) * cg(l2, l2, 0, q2, -q2, 0)
                            emit(k, u, A0(n0p, l0, q0), A(n1, l, m, n1p, l1, q1), A(n2, l, -m, n2p, l2, q2))
            k += 1
        for b, _ in self.clu.get((4, 1), []):
            n, p, l, q, L = b[0:3], b[3:7], b[7:10], b[10:14], b[14]
            mag = [(q0, M - q0, q2, -M - q2, cg(q[0], q[1], L, q0, M - q0, M) * cg(q[2], q[3], L, q2, -M - q2, -M) * cg(L, L, 0, M, -M, 0))
                   for M in range(-L, L + 1) for q0 in range(-q[0], q[0] + 1) if abs(M - q0) <= q[1]
                   for q2 in range(-q[2], q[2] + 1) if abs(M + q2) <= q[3]]
            for m1 in range(-l[0], l[0] + 1):
                for m2 in range(-l[1], l[1] + 1):
                    m3 = -m1 - m2
                    if abs(m3) <= l[2]:
                        c = cg(l[0], l[1], l[2], m1, m2, -m3) * cg(l[2], l[2], 0, m3, -m3, 0)
                        for q0, q1, q2, q3, cm in mag:
                            emit(k, c * cm, A0(p[0], q[0], q0), A(n[0], l[0], m1, p[1], q[1], q1),
                                 A(n[1], l[1], m2, p[2], q[2], q2), A(n[2], l[2], m3, p[3], q[3], q3))
            k += 1
        self.idx = torch.tensor(list(idx), device=self.dev)  # [T, 4]
        self.U = torch.sparse_coo_tensor(torch.tensor([t_of, k_of]), torch.tensor(u_of, dtype=torch.float64), (len(idx), k)).coalesce().to(self.dev)
        c1 = [[v for _, v in self.clu[1, d]] for d in range(1, self.nd + 1)]
        c = [[v for o in (2, 3, 4) for _, v in self.clu.get((o, d), [])] for d in range(1, self.nd + 1)]
        self.c1 = torch.tensor(c1, device=self.dev, dtype=torch.float64)  # [nd, n1]
        self.set(torch.tensor(c, device=self.dev, dtype=torch.float64))

    def set(self, c):
        self.c = c
        self.w = torch.sparse.mm(self.U, c.T)  # [T, nd]

    def features(self, u, mj, mi, first, count):
        """Z (real, imaginary) [columns, atoms] and B1 [atoms, n1] of atoms with `count` pairs each from `first` on."""
        n, J = len(count), int(count.max())
        at = torch.arange(J, device=self.dev)[None, :]
        live = at < count[:, None]
        p = torch.where(live, first[:, None] + at, torch.zeros_like(at))

        def gather(v):  # per pair -> per atom and slot, zero where there is no pair
            return torch.where(live.reshape(live.shape + (1,) * (v.dim() - 1)), v[p], torch.zeros((), dtype=v.dtype, device=v.device))

        r, mu, mui = u.norm(dim=1), mj.norm(dim=1), mi.norm(dim=1)
        fa, fm, fi = self._spline(self.tab_a, r, RCUT), self._spline(self.tab_m, mu, RCUT_M), self._spline(self.tab_m, mui, RCUT_M)
        yr, yi = self._harmonics(u / r[:, None], self.l3a)
        sr, si = self._harmonics(mj / mu[:, None], self.l2m)
        tr, ti = self._harmonics(mi / mui[:, None], self.l2m)
        la = [l for l in range(self.l3a + 1) for _ in range(2 * l + 1)]
        lm = [l for l in range(self.l2m + 1) for _ in range(2 * l + 1)]
        R = fa[:, self.nba:].reshape(-1, self.l3a + 1, self.nr3a)[:, la].transpose(1, 2)  # [P, n, lm]
        M = fm[:, self.nbm:].reshape(-1, self.l2m + 1, self.nr2m)[:, lm].transpose(1, 2)  # [P, n', l'm']
        Mi = fi[:, self.nbm:].reshape(-1, self.l2m + 1, self.nr2m)[:, lm].transpose(1, 2)
        ls3 = (self.l3m + 1) ** 2
        Hr, Hi = M * sr[:, None], M * si[:, None]
        H3 = [v[:, :self.nr3m, :ls3].reshape(len(r), -1) for v in (Hr, Hi)]
        left = [gather((R * v[:, None]).reshape(len(r), -1)).transpose(1, 2) for v in (yr, yi)]
        right = [gather(v) for v in H3]
        Ar = torch.matmul(left[0], right[0]) - torch.matmul(left[1], right[1])
        Ai = torch.matmul(left[0], right[1]) + torch.matmul(left[1], right[0])
        g = gather(fa[:, :self.nba]).transpose(1, 2)
        A2 = [torch.matmul(g, gather(v.reshape(len(r), -1))).reshape(n, -1) for v in (Hr, Hi)]
        A0 = [(Mi * v[:, None]).reshape(n, -1) for v in (tr, ti)]
        o = torch.ones(n, 1, dtype=torch.float64, device=self.dev)
        Zr, Zi = torch.cat([Ar.reshape(n, -1), A2[0], A0[0], o], 1), torch.cat([Ai.reshape(n, -1), A2[1], A0[1], 0 * o], 1)
        return Zr.T.contiguous(), Zi.T.contiguous(), fi[:, :self.nbm] - 1

    def products(self, Zr, Zi):
        """Re prod_s Z[idx_ts]: [T, atoms]."""
        g = lambda s: (Zr[self.idx[:, s]], Zi[self.idx[:, s]])  # noqa: E731
        mul = lambda a, b: (a[0] * b[0] - a[1] * b[1], a[0] * b[1] + a[1] * b[0])  # noqa: E731
        a, b = mul(g(0), g(1)), mul(g(2), g(3))
        return a[0] * b[0] - a[1] * b[1]

    def energies(self, u, mj, mi, first, count):
        Zr, Zi, B1 = self.features(u, mj, mi, first, count)
        rho = (self.w.T @ self.products(Zr, Zi)).T + B1 @ self.c1.T  # [atoms, nd]
        if self.nfemb == 0:
            return rho.sum(1)
        E = 0
        for d in range(self.nd):
            s, pre, m = rho[:, d], self.par[1, d + 1], self.par[2, d + 1]
            y = 10.0 * s * s
            g = torch.where(y > 30.0, torch.zeros_like(y), torch.exp(-y))
            E = E + pre * torch.sign(s) * (((1 - g) * s.abs()) ** m + m * g * s.abs())
        return E

    def chunks(self, off, most):
        """Ranges of atoms of at most `most` each."""
        n = len(off) - 1
        return [(a, min(n, a + most)) for a in range(0, n, most)]

    def evaluate(self, L):
        """eout, flist, tlist, tlist0 of acelib_ for device lists L."""
        off = L["offsets"].long()
        u = L["elist"].reshape(-1, 3) * L["dlist"][:, None]
        mj = L["elist_mom"].reshape(-1, 3) * L["dlist_mom"][:, None]
        mi = L["elist_momi"].reshape(-1, 3) * L["dlist_momi"][:, None]
        most = max(1, int(2e7 / len(self.idx)))
        out = [[], [], [], []]
        for a, b in self.chunks(off, most):
            p0, p1 = int(off[a]), int(off[b])
            x = [t.detach().clone().requires_grad_(True) for t in (u[p0:p1], mj[p0:p1], mi[a:b])]
            E = self.energies(*x, off[a:b] - p0, off[a + 1:b + 1] - off[a:b])
            g = torch.autograd.grad(E.sum(), x)
            for o, v in zip(out, (E.detach(), *g)):
                o.append(v)
        return dict(zip(("eout", "flist", "tlist", "tlist0"), (torch.cat(o) for o in out)))

    def buffers(self, L):
        """evaluate() in arrays with room for MOST pairs an atom."""
        o = self.evaluate(L)
        rest = torch.zeros(MOST * len(o["eout"]) - len(o["flist"]), 3, dtype=torch.float64, device=self.dev)
        return dict(o, flist=torch.cat([o["flist"], rest]), tlist=torch.cat([o["tlist"], rest]))

    def coefficients_gradient(self, L, gE, gF):
        """d/dc of sum_i gE_i E_i + sum_j gF_j . F_j (E linear in c): sum_i gE_i B_i - D_u B_i along u = gF."""
        off, nl = L["offsets"].long(), L["nlist"].long()
        u = L["elist"].reshape(-1, 3) * L["dlist"][:, None]
        mj = L["elist_mom"].reshape(-1, 3) * L["dlist_mom"][:, None]
        mi = L["elist_momi"].reshape(-1, 3) * L["dlist_momi"][:, None]
        count = off[1:] - off[:-1]
        owner = torch.repeat_interleave(torch.arange(len(count), device=self.dev), count)
        du = gF[owner] - gF[nl]
        M, M1 = 0, 0
        for a, b in self.chunks(off, max(1, int(8e6 / len(self.idx)))):
            p0, p1 = int(off[a]), int(off[b])

            def f(x):
                Zr, Zi, B1 = self.features(x, mj[p0:p1], mi[a:b], off[a:b] - p0, count[a:b])
                return self.products(Zr, Zi), B1

            (P, B1), (dP, _) = torch.func.jvp(f, (u[p0:p1],), (du[p0:p1],))
            M = M + P @ gE[a:b] - dP.sum(1)
            M1 = M1 + B1.T @ gE[a:b]
        return torch.cat([M1, torch.sparse.mm(self.U.transpose(0, 1), M[:, None])[:, 0]])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("neigh", "md"):
        return None
    state = prepare(case, seed)
    X = _Exact(_text(case["header"]))
    if kind in ("eval", "host"):
        return X.buffers(state["L"])
    b, c = state["batch"], state["c"].detach()
    n1 = X.c1.shape[1]
    X.c1 = c[None, :n1]
    X.set(c[None, n1:])
    o = X.evaluate(b.L)
    L = b.L
    off = L["offsets"].long()
    owner = torch.repeat_interleave(torch.arange(b.natom, device=c.device), off[1:] - off[:-1])
    struct = b.atom_struct.long()
    F = torch.zeros(b.natom, 3, dtype=torch.float64, device=c.device).index_add(0, owner, -o["flist"]).index_add(0, L["nlist"].long(), o["flist"])
    E = torch.zeros(b.nstruc, dtype=torch.float64, device=c.device).index_add(0, struct, o["eout"])
    gE, gF = 2 * state["weight"] ** 2 * (E - state["E0"]), 2 * (F - state["F0"])
    return dict(E=E, F=F, grad=X.coefficients_gradient(L, gE[struct], gF))
