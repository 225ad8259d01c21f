"""Distances and moments that are not numbers are reported as input errors in every precision, as the reference
stops on them (its table index of a NaN is below the first row), and leave nothing behind; an infinite distance is
a pair beyond the cutoff, whose contribution is zero."""
import numpy as np
import pytest

from helpers import PKG, write_potential

capi, systems = PKG.capi, PKG.systems
torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU visible", allow_module_level=True)

KEYS = ("eout", "flist", "tlist", "tlist0")


@pytest.mark.parametrize("header", ["HTINY", "H500", "HFE", "H500ND2"])
@pytest.mark.parametrize("precision", ["FP64", "MIXED", "MIXED_ACC"])
def test_values_that_are_no_numbers(tmp_path, header, precision):
    capi.init_file(write_potential(str(tmp_path / "p.in"), header, 91))
    s = systems.make_system(2, 92, "uniform")
    a = systems.pack_acelib(s["pos"], s["cell"], s["sdir"], s["smag"], 5.0)
    capi.set_precision(getattr(capi, precision))
    good = capi.acelib(a)
    for key, place in (("dlist", 5), ("dlist_mom", 70), ("dlist_momi", 3)):
        bad = dict(a, **{key: np.array(a[key], dtype=np.float64)})
        bad[key][place] = np.nan
        with pytest.raises(capi.MagaceError, match="small distance" if key == "dlist" else "oment"):
            capi.acelib(bad)
        again = capi.acelib(a)
        for k in KEYS:
            assert np.array_equal(good[k], again[k]), (key, k)
    far, beyond = (dict(a, dlist=np.array(a["dlist"], dtype=np.float64)) for _ in range(2))
    far["dlist"][5], beyond["dlist"][5] = np.inf, 100.0
    far, beyond = capi.acelib(far), capi.acelib(beyond)
    for k in KEYS:
        assert np.array_equal(far[k], beyond[k]), k
    capi.set_precision(capi.FP64)
