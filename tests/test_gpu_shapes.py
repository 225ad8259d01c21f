"""Evaluations at the edges of the kernels' tiles: odd and tiny atom counts (the FP32 adjoint takes two
atoms a workgroup) and neighbour counts of 0, 1 and around the multiples of 16, 32 and 64 that the
density and the forces work in, for headers whose adjoint plans differ (workgroups of 4, 8 and 16
waves) and for every shape class.  Compared with the oracle: FP64 within 1e-10, mixed within 1e-4, the
bars of the golden cases, relative to each output's largest value."""
import sys

import numpy as np
import pytest

from helpers import HEADERS, PKG, relerr, write_potential

capi, systems = PKG.capi, PKG.systems
torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU visible", allow_module_level=True)

import oracle as O  # noqa: E402

# thirteen atomic and five magnetic radial functions at lmax 6 with nine magnetic columns: the largest tables of
# the forces, whose workgroups have two waves in FP64
HEADERS["HLDS"] = dict(PKG.potgen.H6W, nb_a=13, nb_m=5, nr2_m=5, nr3_a=1, nr4_a=1)


def cut_list(counts, seed):
    """acelib_ arrays of len(counts) atoms with counts[i] neighbours each, taken from a bcc list with
    pairs up to 7.0 A (those beyond the cutoff contribute zero)."""
    rng = np.random.default_rng(seed)
    s = systems.make_system(3, seed, "uniform", rcut=7.0)
    a = systems.pack_acelib(s["pos"], s["cell"], s["sdir"], s["smag"], 7.0)
    off, keep = a["offsets"], []
    for i, n in enumerate(counts):
        assert n <= off[i + 1] - off[i]
        keep.append(off[i] + np.sort(rng.choice(off[i + 1] - off[i], n, replace=False)))
    k = np.concatenate(keep).astype(int)
    new = np.concatenate([[0], np.cumsum(counts)])
    N = len(counts)
    out = dict(natom=N, nall=N, nstart=(new[:-1] + 1).astype(np.int32), nstop=new[1:].astype(np.int32),
               nlist=a["nlist"][k], occ=np.ones(N, np.int32), occlist=np.ones(len(k), np.int32))
    for key in ("dlist", "dlist_mom"):
        out[key] = np.ascontiguousarray(a[key][k])
    for key in ("elist", "elist_mom"):
        out[key] = np.ascontiguousarray(a[key].reshape(-1, 3)[k]).reshape(-1)
    out["dlist_momi"] = a["dlist_momi"][:N].copy()
    out["elist_momi"] = a["elist_momi"][:3 * N].copy()
    out["offsets"] = new
    return out


COUNTS = ([57], [0, 1], [15, 16, 17], [31, 32, 33, 47, 48], [63, 64, 65, 0, 100, 2, 58])


@pytest.mark.parametrize("header", ["HTINY", "H500", "H2000", "HFE", "H6W", "H4W", "H500M0", "H500CORE", "HLDS"])
@pytest.mark.parametrize("counts", COUNTS, ids=lambda c: "-".join(map(str, c)))
def test_edges_of_tiles(header, counts, tmp_path):
    pot = write_potential(str(tmp_path / "p.in"), header, 77)
    capi.init_file(pot)
    a = cut_list(counts, 5)
    ref = O.Oracle.load(pot).acelib(a)
    for prec, bar in ((capi.FP64, 1e-10), (capi.MIXED, 1e-4), (capi.MIXED_ACC, 1e-4)):
        capi.set_precision(prec)
        print("shapes: %s %s precision %d" % (header, counts, prec))
        sys.stdout.flush()
        got = capi.acelib(a)
        for k in ("eout", "flist", "tlist", "tlist0"):
            e = relerr(got[k], ref[k])
            assert e <= bar, (k, prec, e)
    capi.set_precision(capi.FP64)
