"""acelib_ calls so small that they always cross in one stream (one chunk at any chunk size) against the device-pointer
entry, which copies nothing: the same kernels on the same atoms, so equal bit for bit.  Sizes: no pairs, one,
outputs and inputs that end in half a 16-byte slot (odd counts) and in a whole one, after a larger call whose values lie in the
staging buffers, into arrays of NaN."""
import numpy as np
import pytest

from helpers import PKG, write_potential

capi, systems = PKG.capi, PKG.systems
torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU visible", allow_module_level=True)

KEYS = ("eout", "flist", "tlist", "tlist0")
INPUTS = ("dlist", "elist", "dlist_momi", "elist_momi", "dlist_mom", "elist_mom")


@pytest.fixture(scope="module")
def whole(tmp_path_factory):
    capi.init_file(write_potential(str(tmp_path_factory.mktemp("one") / "p.in"), "H500", 61))
    s = systems.make_system(4, 62, "uniform")  # 128 atoms
    return systems.pack_acelib(s["pos"], s["cell"], s["sdir"], s["smag"], 5.0)


def first(a, counts):
    """The first len(counts) atoms with their first counts[i] pairs."""
    off = np.asarray(a["offsets"])
    k = np.concatenate([np.arange(off[i], off[i] + n) for i, n in enumerate(counts)]).astype(int)
    n, ends = len(counts), np.cumsum(counts)
    out = dict(natom=n, nall=n, nstart=(ends - counts + 1).astype(np.int32), nstop=ends.astype(np.int32),
               nlist=np.ascontiguousarray(a["nlist"][k]), occ=np.ones(n, np.int32), occlist=np.ones(len(k), np.int32),
               offsets=np.concatenate([[0], ends]).astype(np.int32))
    for key in ("dlist", "dlist_mom"):
        out[key] = np.ascontiguousarray(a[key][k])
    for key in ("elist", "elist_mom"):
        out[key] = np.ascontiguousarray(np.asarray(a[key]).reshape(-1, 3)[k]).reshape(-1)
    out["dlist_momi"] = np.ascontiguousarray(a["dlist_momi"][:n])
    out["elist_momi"] = np.ascontiguousarray(np.asarray(a["elist_momi"]).reshape(-1)[:3 * n])
    return out


def on_the_device(a):
    t = lambda x: torch.as_tensor(np.ascontiguousarray(x), device="cuda")  # noqa: E731
    ins = [t(a["offsets"])] + [t(a[k]) for k in INPUTS]
    N, P = a["natom"], len(a["dlist"])
    outs = [torch.full((n,), np.nan, dtype=torch.float64, device="cuda") for n in (N, 3 * P, 3 * P, 3 * N)]
    stream = torch.cuda.current_stream().cuda_stream
    capi.compute_device(N, P, *[x.data_ptr() for x in ins], *[x.data_ptr() for x in outs], stream=stream)
    capi.check_errors(stream)
    return {k: o.cpu().numpy() for k, o in zip(KEYS, outs)}


@pytest.mark.parametrize("counts", [[0], [1], [57], [2, 1], [0, 0, 0], [33, 34, 33], [1] * 5, [57] * 3, [58] * 4], ids=str)
@pytest.mark.parametrize("precision", ["FP64", "MIXED", "MIXED_ACC"])
def test_equal_to_the_device_entry(whole, counts, precision):
    capi.set_precision(getattr(capi, precision))
    capi.acelib(whole)
    a = first(whole, np.array(counts))
    print("one stream:", counts, precision, flush=True)
    N, P = a["natom"], len(a["dlist"])
    host = capi.acelib(a, dict(_buffers=tuple(np.full(max(n, 1), np.nan) for n in (N, 3 * P, 3 * P, 3 * N))))
    device = on_the_device(a)
    for k, n in zip(KEYS, (N, 3 * P, 3 * P, 3 * N)):
        got = np.asarray(host[k]).reshape(-1)
        assert got.size == n and np.array_equal(got, device[k]), (counts, precision, k)
    capi.set_precision(capi.FP64)
