"""Boxes narrower than twice the list radius: every atom lists nearly all others,
up to a box length apart."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _lj(x, rc):
    d = x[:, None] - x[None]
    r2 = (d * d).sum(2)
    np.fill_diagonal(r2, np.inf)
    i6 = np.where(r2 < rc * rc, 1.0 / r2 ** 3, 0.0)
    return ((24.0 * i6 * (2.0 * i6 - 1.0) / r2)[:, :, None] * d).sum(1)


@pytest.mark.parametrize("precision,tol", [("fp32", 2e-5), ("mixed", 2e-5), ("fp64", 1e-12)])
@pytest.mark.parametrize("walls", [True, False])
@pytest.mark.parametrize("n,density", [(8, 0.15), (12, 0.3), (27, 0.8), (64, 0.8), (130, 0.8), (300, 0.8)])
def test_forces_match_fp64(pkg, n, density, walls, precision, tol):
    L = pkg.synth.box_side(n, density)
    x = pkg.synth.lattice_positions(n, L, 3)
    v = pkg.synth.gaussian_velocities(n, 1.0, 3)
    # without walls the frame is wider than lo .. hi, so a narrower one is named
    hi = L if walls or n > 64 else 0.45 * L
    apl = 2 if n % 2 == 0 else 3
    sim = pkg.Simulation(n, pkg.SimSpec(duration=0, stepwidth=1e-4, rc=2.5, rc_coul=0.0, skin=0.6, rebuild_every=5,
                                        lo=0.0, hi=hi, precision=precision, energy_every=1, atomsperleaf=apl,
                                        walls=walls))
    sim.set_state(x, v, np.zeros(n))
    sim.run(12)
    x, _, f = sim.get_state()
    want = _lj(x, 2.5)
    # FP32 pair terms: some 20 roundings of 2^-24 of terms up to a few times the largest force
    assert np.abs(f - want).max() <= tol * max(1.0, np.abs(want).max())
