"""Lists at radii far outside a dynamics run's."""
import time

import numpy as np
import pytest
from conftest import bruteforce_np, pairs_to_rows, rows_canonical

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pred", [0, 1])
@pytest.mark.parametrize("r", [-1.0, -1e-30, -1e30, 0.0])
def test_radii_without_pairs_take_no_time(pkg, r, pred):
    """No distance is below such a radius: sqrt(s) < r holds nowhere, and s < r r
    (the other predicate) only with r r > 0.  A threshold searched for float by
    float from r r down to 0 took 6 s at r = -1; a call takes under 1 ms."""
    n = 300
    x = pkg.synth.uniform_positions(n, 6.0, 3).astype(np.float32)
    spec = pkg.SpheresBVHSpecs(neighbor_distance=r, atom_count=n, atomsperleaf=4)
    pkg.neighborlist_device(x, spec, 0, pkg.MORTON_INTERLEAVE)  # buffers and code are there
    t = time.perf_counter()
    _, count = pkg.neighborlist_device(x, spec, pred, pkg.MORTON_INTERLEAVE)
    assert time.perf_counter() - t < 0.5
    assert pred == 0 or count == 0


@pytest.mark.parametrize("pred", [0, 1])
@pytest.mark.parametrize("n", [64, 1200])
@pytest.mark.parametrize("r", [3e12, 1e18, 5e18, 1e19, 1.8e19])
def test_cell_list_where_squares_overflow(pkg, n, r, pred):
    """Points on a line of some n / 4 radii, near it and around it: squares of
    coordinates overflow where squared distances within the radius do not."""
    rng = np.random.default_rng(n)
    x = rng.random((n, 3)) * [n / 4, 0.2, 0.2]
    x = (x * r).astype(np.float32)
    with np.errstate(over="ignore", invalid="ignore"):
        want = bruteforce_np(x, r, pred)
    got = rows_canonical(pairs_to_rows(pkg.cell_neighborlist(x, r, pred)))
    assert len(want) > 0 and np.array_equal(got, want)
