"""An atom thrown far out by an overlap: its leaf's box spans the system, and
squares about the leaf's centre overflow, but the other atoms' forces are what
they were."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

pytestmark = pytest.mark.gpu


def _lj(x, rc):
    """FP64 Lennard-Jones forces of the pairs closer than rc."""
    i, j = cKDTree(x).query_pairs(rc, output_type="ndarray").T
    d = x[i] - x[j]
    r2 = (d * d).sum(1)
    i6 = 1.0 / r2 ** 3
    p = (24.0 * i6 * (2.0 * i6 - 1.0) / r2)[:, None] * d
    f = np.zeros_like(x)
    np.add.at(f, i, p)
    np.add.at(f, j, -p)
    return f


# leaves of 16 shared by four waves (up to 16,384 atoms) and of 32; dense systems
# (density 4: the walk and the table build apart)
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("n,apl,density", [(63, 3, 0.8), (4100, 5, 0.8), (4100, 4, 4.0), (16641, 3, 0.8),
                                           (20000, 16, 4.0)])
@pytest.mark.parametrize("far", [1e12, 1e20, 1e30])
def test_forces_beside_a_far_atom(pkg, n, apl, density, far, precision):
    L = pkg.synth.box_side(n, density)
    x = pkg.synth.lattice_positions(n, L, 3).astype(np.float32).astype(np.float64)
    x[n // 2] = far
    sim = pkg.Simulation(n, pkg.SimSpec(duration=0, stepwidth=1e-9, rc=2.5, rc_coul=0.0, skin=0.3, rebuild_every=2,
                                        lo=0.0, hi=L, precision=precision, energy_every=1, atomsperleaf=apl,
                                        resort_every=4, walls=False))
    sim.set_state(x, np.zeros((n, 3)), np.zeros(n))
    sim.run(9)  # lists with new keys and in the old order
    x, _, f = sim.get_state()
    keep = np.arange(n) != n // 2
    want = np.zeros((n, 3))
    want[keep] = _lj(x[keep], 2.5)
    # per pair some 20 roundings, of a distance whose 14th power is the steepest term, and sums of at most 400
    # pairs: 1e3 units (lists without the pairs beside the far atom were off by 0.3 to 1 of the largest force)
    tol = 1e3 * (2.0 ** -53 if precision == "fp64" else 2.0 ** -24) * np.abs(want).max()
    assert np.abs(f[keep] - want[keep]).max() < tol
