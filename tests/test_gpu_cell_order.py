"""The cell list's two searches, a lane and a wave per atom, on either side of the
line between them: 131,072 atoms and five atoms a cell.  Both give the pairs of
the definition in one order, by the places of their two atoms in cell order."""
import numpy as np
import pytest
from conftest import pairs_to_rows
from scipy.spatial import cKDTree

pytestmark = pytest.mark.gpu


def _places(x, r):
    """Each atom's place in cell order (the sort is stable) and the number of cells."""
    lo = x.min(0).astype(np.float64)
    ext = x.max(0).astype(np.float64) - lo
    g = np.clip(np.floor(ext / (np.float64(r) * (1.0 + 1e-4))), 1, 1024).astype(np.int64)
    assert g.prod() <= 2 * len(x) + 64
    c = np.minimum(np.floor((x - lo) * (g / ext)), g - 1).astype(np.int64)
    key = (c[:, 2] * g[1] + c[:, 1]) * g[0] + c[:, 0]
    place = np.empty(len(x), np.int64)
    place[np.argsort(key, kind="stable")] = np.arange(len(x))
    return place, int(g.prod())


# lanes: from 131,072 atoms up with fewer than five a cell
@pytest.mark.parametrize("pred", [0, 1])
@pytest.mark.parametrize("n,r,lanes", [(131072, 1.2, True), (131075, 1.5, True), (131072, 1.75, True),
                                       (131071, 1.2, False), (131072, 2.0, False), (200001, 1.3, True)])
def test_pairs_and_order(pkg, n, r, lanes, pred):
    x = pkg.synth.uniform_positions(n, pkg.synth.box_side(n), 3).astype(np.float32)
    r = np.float32(r)
    place, cells = _places(x, r)
    assert (n >= 131072 and n < 5.0 * cells) == lanes
    ij = cKDTree(x).query_pairs(float(r) * 1.001, output_type="ndarray")
    d = x[ij[:, 0]] - x[ij[:, 1]]
    s = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]
    keep = s < r * r if pred == 0 else np.sqrt(s) < r
    ij, s = np.sort(ij[keep], axis=1), s[keep]
    p = np.sort(place[ij], axis=1)
    order = np.lexsort((p[:, 1], p[:, 0]))
    want = np.stack([ij[order, 0], ij[order, 1], np.sqrt(s[order]).view(np.uint32).astype(np.int64)], axis=1)
    assert np.array_equal(pairs_to_rows(pkg.cell_neighborlist(x, r, pred)), want)
