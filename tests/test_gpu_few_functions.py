"""Potentials without some of the products: pair functions only (no magnetic radial function of A, so A has no
columns), no atomic radial function, and the functions of the atoms' own moments alone (no A2 either, an empty feature
vector), in every shape class.  Compared with the oracle: FP64 within 1e-10, mixed within 1e-4, the bars of the
golden cases, relative to each output's largest value; a fit's dE/dc with linear embedding is the oracle's B vectors,
within 1e-10 of the largest."""
import numpy as np
import pytest

from helpers import PKG, relerr

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU visible", allow_module_level=True)

import oracle as O  # noqa: E402

capi, fit, potgen, systems, nbr = PKG.capi, PKG.fit, PKG.potgen, PKG.systems, PKG.neighbors
NO_A = dict(nr3_m=0, nr4_m=0)
FEW = {"pairs-lmax4": dict(potgen.H500, **NO_A), "pairs-lmax6": dict(potgen.H2000, **NO_A),
       "pairs-wide": dict(potgen.HFE, **NO_A), "pairs-medium": dict(potgen.H4W, **NO_A),
       "pairs-tiny": dict(potgen.HTINY, **NO_A), "pairs-l0": dict(potgen.H500, l3m=0, l4m=0, **NO_A),
       "no-atomic-radial": dict(potgen.H500, nr3_a=0, nr4_a=0),
       "moments": dict(potgen.H500, nr2_m=0, **NO_A),
       "moments-l0": dict(potgen.H500, nr2_m=0, l2m=0, nr3_a=0, nr4_a=0, l3a=0, l3m=0, l4a=0, l4m=0, **NO_A)}


def potential(tmp_path, header):
    path = str(tmp_path / "Fe.pbe.in")
    with open(path, "w") as f:
        f.write(potgen.render(header, capi.enumerate_basis(header), 21))
    return path


@pytest.mark.parametrize("name", sorted(FEW))
@pytest.mark.parametrize("cells", [(1, 1, 1), (3, 2, 2)])
def test_evaluation(tmp_path, name, cells):
    path = potential(tmp_path, FEW[name])
    capi.init_file(path)
    rng = np.random.default_rng(22)
    pos, cell = systems.bcc_box(*cells)
    pos = systems.jitter(pos, rng, 0.08)
    a = systems.pack_acelib(pos, cell, *systems.spins_uniform(len(pos), rng), 5.6)
    ref = O.Oracle.load(path).acelib(a)
    for prec, bar in ((capi.FP64, 1e-10), (capi.MIXED, 1e-4), (capi.MIXED_ACC, 1e-4)):
        capi.set_precision(prec)
        print("few functions: %s %s precision %d" % (name, cells, prec), flush=True)
        got = capi.acelib(a)
        for k in ("eout", "flist", "tlist", "tlist0"):
            e = relerr(got[k], ref[k])
            assert e <= bar, (k, prec, e)
    capi.set_precision(capi.FP64)


@pytest.mark.parametrize("name", ["pairs-lmax4", "pairs-wide", "pairs-medium", "no-atomic-radial"])
def test_fit_gradient(tmp_path, name):
    h = dict(FEW[name], nfemb=0)
    path = potential(tmp_path, h)
    capi.init_file(path)
    rng = np.random.default_rng(23)
    structs = []
    for cells in ((2, 1, 1), (2, 2, 1)):
        pos, cell = systems.bcc_box(*cells)
        sdir, smag = systems.spins_uniform(len(pos), rng)
        structs.append(dict(pos=systems.jitter(pos, rng, 0.08), cell=cell, sdir=sdir, smag=smag))
    batch = fit.Batch(structs, 5.0)
    gE = rng.normal(size=len(structs))
    o = O.Oracle.load(path)
    want = sum(w * o.bvectors(nbr.neilist(s["pos"], s["sdir"] * s["smag"][:, None], s["cell"], 5.0)).sum(axis=0)
               for s, w in zip(structs, gE))
    print("few functions: fit", name, flush=True)
    batch.forward(torch.zeros(len(structs), dtype=torch.float64, device="cuda"),
                  torch.zeros(batch.natom, 3, dtype=torch.float64, device="cuda"))
    g = torch.zeros(capi.fit_ncoef(), dtype=torch.float64, device="cuda")
    batch.backward(torch.tensor(gE, device="cuda"), torch.zeros(batch.natom, 3, dtype=torch.float64, device="cuda"), g)
    assert np.abs(g.cpu().numpy() - want).max() <= 1e-10 * np.abs(want).max()
