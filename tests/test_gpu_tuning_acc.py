"""The density's variants belong to the accumulation recipe: every (variant, neighbour split) candidate matches the
reference's golden vectors there, to the 1e-5 that the recipe keeps on forces elsewhere; FP64 and mixed evaluations
do not change by a bit with the setting, and tuning in these precisions leaves the recipe's setting alone."""
import numpy as np
import pytest

from helpers import PKG, load_case, relerr, write_potential

capi, systems = PKG.capi, PKG.systems
torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU visible", allow_module_level=True)

KEYS = ("eout", "flist", "tlist", "tlist0")


@pytest.mark.parametrize("name", ["h500_128", "h2000_16", "hfe_16", "h6w_16", "h4w_16"])
def test_candidates(name, tmp_path):
    c = load_case(name, tmp_path)
    capi.init_file(c["pot"])
    for precision in (capi.FP64, capi.MIXED):
        capi.set_precision(precision)
        first = None
        for cand in ((-1, 0),) + capi.TUNE_CANDIDATES:
            capi.set_tuning(fp64=cand, mixed=cand)
            got = capi.acelib(c["a"])
            first = first or got
            for k in KEYS:
                assert np.array_equal(got[k], first[k]), (name, precision, cand, k)
    capi.set_precision(capi.MIXED_ACC)
    for cand in ((-1, 0),) + capi.TUNE_CANDIDATES:
        capi.set_tuning(mixed=cand)
        got = capi.acelib(c["a"])
        for k in KEYS:
            e = relerr(got[k], c["ref"][k])
            assert e <= 1e-5, (name, cand, k, e)
    capi.set_precision(capi.FP64)


def test_tune(tmp_path):
    capi.init_file(write_potential(str(tmp_path / "p.in"), "H500", 2027))
    s = systems.make_system(8, 3, "uniform")
    a = systems.pack_acelib(s["pos"], s["cell"], s["sdir"], s["smag"], 5.0)
    t = lambda x, dt=torch.float64: torch.as_tensor(np.ascontiguousarray(x), dtype=dt, device="cuda")
    N, P = a["natom"], len(a["dlist"])
    ins = [t(a["offsets"], torch.int32)] + [t(a[k]) for k in ("dlist", "elist", "dlist_momi", "elist_momi",
                                                                "dlist_mom", "elist_mom")]
    outs = [torch.zeros(n, dtype=torch.float64, device="cuda") for n in (N, 3 * P, 3 * P, 3 * N)]
    tune = lambda: capi.tune(N, P, *[x.data_ptr() for x in ins], *[o.data_ptr() for o in outs], reps=3,  # noqa: E731
                             stream=torch.cuda.current_stream().cuda_stream)
    for setting in (dict(fp64=(1, 3), mixed=(2, 4)), dict()):
        capi.set_tuning(**setting)
        kept = capi.get_tuning()
        for precision in (capi.FP64, capi.MIXED):
            capi.set_precision(precision)
            best, ms = tune()
            assert best == kept[precision == capi.MIXED] and capi.get_tuning() == kept
            assert len(set(ms.values())) == 1 and ms[0, 0] > 0
    capi.set_precision(capi.MIXED_ACC)
    best, ms = tune()
    assert best in capi.TUNE_CANDIDATES and ms[best] > 0
    assert all(v is None or v >= ms[best] for v in ms.values())
    assert capi.get_tuning() == (kept[0], best)
    capi.set_precision(capi.FP64)
