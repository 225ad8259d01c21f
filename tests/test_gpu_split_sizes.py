"""FP64 evaluations at the line from which they run as two halves on two streams (12288 atoms): one atom below it, at it
and above it, odd counts included, against the same evaluation in one sequence.  The same kernels work on the same
atoms, so results are equal bit for bit."""
import os

import numpy as np
import pytest

from helpers import PKG, write_potential

capi, systems, neighbors = PKG.capi, PKG.systems, PKG.neighbors
torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU visible", allow_module_level=True)


def evaluate(L, natom, split, monkeypatch):
    monkeypatch.setenv("MAGACE_SPLIT_STREAMS", split)
    out = [torch.full((n,), np.nan, dtype=torch.float64, device="cuda") for n in (natom, 3 * L["npairs"], 3 * L["npairs"], 3 * natom)]
    capi.compute_device(natom, L["npairs"], *(L[k].data_ptr() for k in ("offsets", "dlist", "elist", "dlist_momi", "elist_momi",
                                                                      "dlist_mom", "elist_mom")),
                        *(o.data_ptr() for o in out), torch.cuda.current_stream().cuda_stream)
    capi.check_errors(torch.cuda.current_stream().cuda_stream)
    return out


@pytest.mark.parametrize("natom", [12287, 12288, 12289, 13999])
def test_two_halves_equal_one_sequence(tmp_path, monkeypatch, natom):
    capi.init_file(write_potential(str(tmp_path / "p.in"), "H500", 80))
    rng = np.random.default_rng(81)
    pos, cell = systems.bcc_box(20, 20, 18)
    pos = systems.jitter(pos[:natom], rng, 0.05)
    sdir, smag = systems.spins_uniform(natom, rng)
    nb = neighbors.DeviceNeighbors(np.array([natom], np.int32), [1], cell[None], 5.0)
    L = nb.build(torch.tensor(pos, device="cuda"), torch.tensor(sdir * smag[:, None], device="cuda"))
    one, two = evaluate(L, natom, "0", monkeypatch), evaluate(L, natom, "1", monkeypatch)
    for a, b in zip(one, two):
        assert torch.equal(a, b)
