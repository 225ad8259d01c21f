"""The gradient in the coefficients for plans of one group of tiles, of many groups and with products of
entries (body orders 5 and 6), one and two densities, for atom counts at the edges of a workgroup's share
(1, 3, 5 and more atoms).  With linear embedding dE/dc is the oracle's B vectors, within 1e-10 of the
largest as in the other fits, and the forces' part is their derivative along the displacements, by central
differences with steps of 1e-4 and 2e-4 A, extrapolated: against lengths of 0.3 A their error is below
1e-6, and the sums' own rounding (1e-15 of their largest value) enters as (4 + 1/2) / 3 of it over the
step, which is all that one atom and its images have, whose derivative is 0."""
import numpy as np
import pytest

from helpers import HEADERS, PKG

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU visible", allow_module_level=True)

import oracle as O  # noqa: E402

capi, fit, potgen, systems, nbr = PKG.capi, PKG.fit, PKG.potgen, PKG.systems, PKG.neighbors
SIZES = {1: ((1, 1, 1, 1),), 3: ((2, 1, 1, 1),), 5: ((1, 1, 1, 0), (2, 1, 1, 1)), 35: ((2, 2, 2, 1), (3, 2, 1, 0), (2, 1, 2, 0))}


def structures(natom, seed):
    rng = np.random.default_rng(seed)
    out = []
    for n1, n2, n3, vac in SIZES[natom]:
        pos, cell = systems.bcc_box(n1, n2, n3)
        pos = systems.jitter(pos[vac:], rng, 0.08)
        sdir, smag = systems.spins_uniform(len(pos), rng)
        out.append(dict(pos=pos, cell=cell, sdir=sdir, smag=smag))
    assert sum(len(s["pos"]) for s in out) == natom
    return out


def bsum(o, structs, weights, shift=0.0, u=None):
    """Weighted sum of the structures' B vectors, atoms moved by shift * u."""
    want, a0 = np.zeros(sum(o.counts())), 0
    for s, w in zip(structs, weights):
        n = len(s["pos"])
        pos = s["pos"] + (shift * u[a0:a0 + n] if u is not None else 0.0)
        want += w * o.bvectors(nbr.neilist(pos, s["sdir"] * s["smag"][:, None], s["cell"], 5.0)).sum(axis=0)
        a0 += n
    return want


@pytest.mark.parametrize("header", ["HTINY", "H500ND2", "H2000", "HFE", "H4W", "H56"])
@pytest.mark.parametrize("natom", sorted(SIZES))
def test_gradient_of_energies_and_forces(tmp_path, header, natom):
    h = dict(HEADERS[header], nfemb=0)
    pot = str(tmp_path / "Fe.pbe.in")
    with open(pot, "w") as f:
        f.write(potgen.render(h, capi.enumerate_basis(h), 31, c_scale=1e-2))
    capi.init_file(pot)
    structs = structures(natom, 4)
    batch = fit.Batch(structs, 5.0)
    rng = np.random.default_rng(5)
    gE, u = rng.normal(size=len(structs)), rng.normal(size=(natom, 3))
    o = O.Oracle.load(pot)
    nd = int(h.get("ndensity", 1))
    cuts = np.cumsum([0] + list(o.counts()))
    step = 1e-4
    still = bsum(o, structs, 1 + 0 * gE)
    def slope(k):
        return (bsum(o, structs, 1 + 0 * gE, k * step, u) - bsum(o, structs, 1 + 0 * gE, -k * step, u)) / (2 * k * step)

    moved = -(4 * slope(1) - slope(2)) / 3
    for wE, gF, want, tol in ((gE, 0 * u, bsum(o, structs, gE), 0.0), (0 * gE, u, moved, 1.5e-15 * np.abs(still).max() / step)):
        tol += (1e-6 if tol else 1e-10) * np.abs(want).max()
        E = torch.zeros(len(structs), dtype=torch.float64, device="cuda")
        F = torch.zeros(natom, 3, dtype=torch.float64, device="cuda")
        g = torch.zeros(capi.fit_ncoef(), dtype=torch.float64, device="cuda")
        batch.forward(E, F)
        batch.backward(torch.tensor(wE, device="cuda"), torch.tensor(gF, device="cuda"), g)
        want = np.concatenate([np.tile(want[cuts[k]:cuts[k + 1]], nd) for k in range(6)])
        err = np.abs(g.cpu().numpy() - want).max()
        assert err <= tol


@pytest.mark.parametrize("header", ["H500", "H500ND2"])
def test_state_serves_backward_as_forward_does(tmp_path, header):
    pot = str(tmp_path / "Fe.pbe.in")
    with open(pot, "w") as f:
        f.write(potgen.render(HEADERS[header], capi.enumerate_basis(HEADERS[header]), 32, c_scale=1e-2))
    capi.init_file(pot)
    structs = structures(35, 6)
    batch = fit.Batch(structs, 5.0)
    rng = np.random.default_rng(7)
    gE, gF = torch.tensor(rng.normal(size=len(structs)), device="cuda"), torch.tensor(rng.normal(size=(35, 3)), device="cuda")
    grads = []
    for forward in (True, False):
        if forward:
            batch.forward(torch.zeros(len(structs), dtype=torch.float64, device="cuda"),
                          torch.zeros(35, 3, dtype=torch.float64, device="cuda"))
        else:
            batch.state()
        g = torch.zeros(capi.fit_ncoef(), dtype=torch.float64, device="cuda")
        batch.backward(gE, gF, g)
        grads.append(g.cpu().numpy())
    # the same sums; those over atoms meet in memory in any order
    assert np.abs(grads[0] - grads[1]).max() <= 1e-12 * np.abs(grads[0]).max()
