"""Neighbour builds at the sizes where the device's route changes: offsets scanned in one launch up to 65536
entries, image candidates counted per tile of 256 and added up by every tile up to 4096 tiles, boxes with more
than 64 atoms, atoms with more than 64 and more than 128 neighbours.  The pairs are compared with a periodic
k-d tree, the offsets with the counts, the distances and shifts with the positions."""
import numpy as np
import pytest

from helpers import PKG

torch = pytest.importorskip("torch")
spatial = pytest.importorskip("scipy.spatial")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU visible", allow_module_level=True)


# cells of bcc with two atoms each: 512 and 513 are either side of a tile of 1024 offsets, 32 is 65536 atoms, 33 more;
# 28 and 29 are either side of 4096 candidate tiles
@pytest.mark.parametrize("n, rcut", [(1, 5.0), (2, 9.0), (8, 5.0), (8, 7.5), (28, 3.0), (29, 3.0), (32, 3.0), (33, 3.0)])
def test_pairs_against_a_tree(n, rcut):
    s = PKG.systems.make_system(n, 3, "uniform")
    pos, L = s["pos"], np.diag(s["cell"])[0]
    nat = len(pos)
    print("neighbours: %d atoms, cutoff %.1f" % (nat, rcut), flush=True)
    most = int(nat * (4.19 * rcut**3 * 2 / 2.8**3 * 1.3 + 30))
    nb = PKG.neighbors.DeviceNeighbors([nat], [1], s["cell"][None], rcut, capacity=most)
    mag = s["sdir"] * s["smag"][:, None]
    for _ in range(2):
        r = nb.build(torch.tensor(pos, device="cuda"), torch.tensor(mag, device="cuda"))
    P = int(r["npairs"])
    off, nl = nb.offsets.cpu().numpy()[:nat + 1], nb.nlist.cpu().numpy()[:P]
    dl, el = nb.dlist.cpu().numpy()[:P], nb.elist.cpu().numpy().reshape(-1, 3)[:P]
    assert off[0] == 0 and off[-1] == P and (np.diff(off) >= 0).all()
    # images of every atom within the cutoff of the cell
    w = pos - np.floor(pos / L) * L
    k = int(np.ceil(rcut / L))
    sh = np.array([(a, b, c) for a in range(-k, k + 1) for b in range(-k, k + 1) for c in range(-k, k + 1)]) * L
    img = (w[None] + sh[:, None]).reshape(-1, 3)
    org = np.tile(np.arange(nat), len(sh))
    near = ((img > -rcut - 1e-6) & (img < L + rcut + 1e-6)).all(1)
    img, org = img[near], org[near]
    m = spatial.cKDTree(w).sparse_distance_matrix(spatial.cKDTree(img), rcut, output_type="coo_matrix")
    keep = m.data > 1e-9  # not an atom with itself
    i, j, d = m.row[keep], org[m.col[keep]], m.data[keep]
    assert P == len(i)
    assert np.array_equal(np.diff(off), np.bincount(i, minlength=nat))
    mine = np.repeat(np.arange(nat), np.diff(off))
    a, b = np.lexsort((d.round(9), j, i)), np.lexsort((dl.round(9), nl, mine))
    assert np.array_equal(i[a], mine[b]) and np.array_equal(j[a], nl[b])
    # positions of a few angstrom to a hundred, so rounding of 1e-14 relative and a sum of two squares
    assert np.abs(d[a] - dl[b]).max() <= 1e-11
    back = pos[mine] - pos[nl] - dl[:, None] * el
    assert np.abs(back / L - np.round(back / L)).max() <= 1e-11
