"""acelib_ calls that cross in one stream (one chunk, up to 4 MiB of inputs) against the same calls cut in chunks
of 1024 pairs and copied by the three-stream pipeline: the same kernels on the same atoms, so equal bit for
bit.  Sizes: pair counts that end a 16-byte slot or not, no pairs, both sides of the 4 MiB line.  An error
reported by one call is not reported by the next."""
import os

import numpy as np
import pytest

from helpers import PKG, write_potential

capi, systems = PKG.capi, PKG.systems
torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU visible", allow_module_level=True)

KEYS = ("eout", "flist", "tlist", "tlist0")


@pytest.fixture(scope="module")
def whole(tmp_path_factory):
    capi.init_file(write_potential(str(tmp_path_factory.mktemp("small") / "p.in"), "H500", 78))
    s = systems.make_system(9, 79, "uniform")  # 1458 atoms
    return systems.pack_acelib(s["pos"], s["cell"], s["sdir"], s["smag"], 5.0)


def cut(a, natom, pairs):
    """The first natom atoms with the first pairs of each left out until `pairs` are left."""
    off = np.asarray(a["offsets"])[:natom + 1]
    k = np.arange(off[-1])[off[-1] - pairs:] if pairs <= off[-1] else np.arange(off[-1])
    new = np.searchsorted(k, off)
    out = dict(natom=natom, nall=natom, nstart=(new[:-1] + 1).astype(np.int32), nstop=new[1:].astype(np.int32),
               nlist=np.ascontiguousarray(a["nlist"][k]), occ=np.ones(natom, np.int32), occlist=np.ones(len(k), np.int32))
    for key in ("dlist", "dlist_mom"):
        out[key] = np.ascontiguousarray(a[key][k])
    for key in ("elist", "elist_mom"):
        out[key] = np.ascontiguousarray(np.asarray(a[key]).reshape(-1, 3)[k]).reshape(-1)
    out["dlist_momi"] = np.ascontiguousarray(a["dlist_momi"][:natom])
    out["elist_momi"] = np.ascontiguousarray(np.asarray(a["elist_momi"]).reshape(-1)[:3 * natom])
    return out


def both(a):
    one = capi.acelib(a)
    os.environ["MAGACE_ACELIB_CHUNK_PAIRS"] = "1024"
    try:
        return one, capi.acelib(a)
    finally:
        del os.environ["MAGACE_ACELIB_CHUNK_PAIRS"]


@pytest.mark.parametrize("natom,pairs", [(1, 0), (1, 57), (2, 3), (3, 100), (40, 2049), (41, 2050), (1130, 10 ** 9), (1140, 10 ** 9)])
def test_one_stream_equals_chunks(whole, natom, pairs):
    a = cut(whole, natom, pairs)
    for prec in (capi.FP64, capi.MIXED):
        capi.set_precision(prec)
        one, chunks = both(a)
        for k in KEYS:
            assert np.array_equal(np.asarray(one[k]), np.asarray(chunks[k])), (natom, pairs, prec, k)
    capi.set_precision(capi.FP64)


def test_errors_are_reported_once(whole):
    a = cut(whole, 4, 200)
    good = capi.acelib(a)
    bad = dict(a, dlist=a["dlist"].copy())
    bad["dlist"][7] = 1e-5
    with pytest.raises(capi.MagaceError):
        capi.acelib(bad)
    again = capi.acelib(a)
    for k in KEYS:
        assert np.array_equal(np.asarray(good[k]), np.asarray(again[k]))
