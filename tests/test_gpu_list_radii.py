"""Lists at radii far outside a dynamics run's."""
import time

import numpy as np
import pytest

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
