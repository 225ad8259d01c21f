"""Mixed precision with radial coefficients that cancel: the fitted example potential, and potentials whose R_{l,n}
are least-squares fits to narrow functions of the distance, of every kind of plan for them (as many radial functions as base
functions or fewer; more; linearly dependent ones and one that is zero).  Each output's error against 64 bits, root
mean square over root mean square, is at most sixteen roundings to 32 bits (2^-24 each): an output passes through about that many
(radial function, harmonic, magnetic function, their product, the sum over pairs, the pair products, their
sum, the gradient's), and their errors add at most in full.  The linearly dependent ones are fits without regard to the size of
their coefficients (up to 1e9): the oracle's table, in 64 bits, has slopes that differ from those of its own base
functions by more than the bar, so pair forces are not compared there.

In FP64 the fitted potential's results are those of the oracle's table of R, so that only the rounding of sums of some
hundred terms is left: 500 times 2^-52 of each output's largest value."""
import numpy as np
import pytest

from helpers import FE_CASES, HEADERS, PKG, fe_case, fe_example, relerr

capi, potgen, systems = PKG.capi, PKG.potgen, PKG.systems
torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU visible", allow_module_level=True)

import oracle as O  # noqa: E402

BAR = 16 * 2.0 ** -24


def check(a, ref, name, keys=("eout", "flist", "tlist", "tlist0")):
    for precision in (capi.MIXED, capi.MIXED_ACC):
        capi.set_precision(precision)
        got = capi.acelib(a)
        for k in keys:
            e = np.sqrt(np.mean((got[k] - ref[k]) ** 2) / np.mean(ref[k] ** 2))
            print("  %s precision %d %s: %.2e" % (name, precision, k, e), flush=True)
            assert e <= BAR, (name, precision, k, e)
    capi.set_precision(capi.FP64)


@pytest.mark.parametrize("name", ["nc16", "nc128"])
def test_fitted_potential(tmp_path, name):
    path, z = fe_example(tmp_path)
    capi.init_file(path, rcut=float(z["rcut"]), rcut_magnetic=float(z["rcut_magnetic"]), smear=float(z["smear"]))
    check(*fe_case(z, name), name)


@pytest.mark.parametrize("name", FE_CASES)
def test_fitted_potential_fp64(tmp_path, name):
    path, z = fe_example(tmp_path)
    capi.init_file(path, rcut=float(z["rcut"]), rcut_magnetic=float(z["rcut_magnetic"]), smear=float(z["smear"]))
    a, ref = fe_case(z, name)
    got = capi.acelib(a)
    for k in ("eout", "flist", "tlist", "tlist0"):
        e = relerr(got[k], ref[k])
        print("  %s FP64 %s: %.2e" % (name, k, e), flush=True)
        assert e <= 500 * 2.0 ** -52, (name, k, e)


def narrow(h, dependent):
    """crad_atomic [nr3_a][l3a + 1][nb_a] of least-squares fits to Gaussians of 0.35 A width; dependent: the same for
    every l, and none for the last n."""
    r = 5.0 * np.arange(1, 2001) / 2000
    g = np.array([O.radbase(h["radtype_a"], h["lambda_a"], h["nb_a"], h["cut_a"], h["dcut_a"], x)[0] for x in r])
    far = r > 1.9
    c = np.zeros((h["nr3_a"], h["l3a"] + 1, h["nb_a"]))
    for n, centre in enumerate(np.linspace(2.2, 4.2, h["nr3_a"])):
        fit = np.linalg.lstsq(g[far], np.exp(-((r[far] - centre) / 0.35) ** 2), rcond=None)[0]
        for l in range(h["l3a"] + 1):
            c[n, l] = fit if dependent else fit * (1 + 0.1 * l) * (1 + 0.01 * np.cos(np.arange(h["nb_a"]) * (n + 1) * (l + 2)))
    if dependent:
        c[-1] = 0.0
    return c


@pytest.mark.parametrize("dependent", [False, True])
@pytest.mark.parametrize("header", ["HTINY", "H500", "H2000", "HFE", "H4W", "H6W"])
def test_cancelling_coefficients(tmp_path, header, dependent):
    h = HEADERS[header]
    basis = capi.enumerate_basis(h)
    rng = np.random.default_rng(51)
    values = dict(crad_a=narrow(h, dependent), crad_m=rng.normal(size=(h["nr2_m"], h["l2m"] + 1, h["nb_m"])) / np.sqrt(h["nb_m"]),
                  c={k: rng.normal(0.0, 1e-2, len(basis[k])) for k in basis})
    path = str(tmp_path / "Fe.pbe.in")
    with open(path, "w") as f:
        f.write(potgen.render(h, basis, 0, values=values))
    capi.init_file(path)
    s = systems.make_system(3, 52, "uniform")
    a = systems.pack_acelib(s["pos"], s["cell"], s["sdir"], s["smag"], 5.0)
    check(a, O.Oracle.load(path).acelib(a), header, ("eout", "tlist", "tlist0") if dependent else ("eout", "flist", "tlist", "tlist0"))
