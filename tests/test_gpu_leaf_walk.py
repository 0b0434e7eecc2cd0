"""The list walk over leaves of 32 consecutive atoms and boxes of 64 leaves:
leaf sizes and atom counts that leave its last leaf, chunk or wave ragged, and
enough chunks for the boxes of 64 chunks, against the cell-list walk."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _state(pkg, n, seed):
    L = pkg.synth.box_side(n)
    return L, pkg.synth.lattice_positions(n, L, seed), pkg.synth.gaussian_velocities(n, 1.0, seed), \
        pkg.synth.balanced_charges(n, seed)


def _run(pkg, n, apl, walk, precision, steps, state):
    L, x, v, q = state
    sim = pkg.Simulation(n, pkg.SimSpec(duration=0, stepwidth=0.001, rc=2.5, rc_coul=2.5, skin=0.3, rebuild_every=4,
                                        lo=0.0, hi=L, precision=precision, energy_every=1, atomsperleaf=apl,
                                        resort_every=8, list_walk=walk))
    sim.set_state(x, v, q)
    sim.run(steps)
    return np.array(sim.get_state()[0]), np.array(sim.energies())


# up to 16,384 atoms four waves share each 64: one wave less one atom, one more
# than a workgroup and than a chunk (1,024 or 2,048 atoms), odd leaf sizes
@pytest.mark.parametrize("n,apl", [(2, 1), (63, 3), (66, 2), (257, 1), (2049, 3), (4100, 5), (16383, 3), (16641, 3), (65793, 3)])
def test_ragged_leaves(pkg, n, apl):
    s = _state(pkg, n, n)
    x0, e0 = _run(pkg, n, apl, 0, "fp64", 13, s)
    x3, e3 = _run(pkg, n, apl, 3, "fp64", 13, s)
    # the same pairs summed in another order: 13 steps of FP64 rounding
    assert np.abs(x0 - x3).max() < 1e-11
    assert np.array_equal(e0[:, 4], e3[:, 4])  # pairs inside the cutoff
    assert np.allclose(e0[:, 1:4], e3[:, 1:4], rtol=1e-11, atol=1e-9)


def test_more_chunks_than_are_looked_at_one_by_one(pkg):
    n = 32 * 64 * 512 + 35  # 513 chunks, the last of two leaves
    s = _state(pkg, n, 5)
    x0, e0 = _run(pkg, n, 1, 0, "fp32", 5, s)
    x3, e3 = _run(pkg, n, 1, 3, "fp32", 5, s)
    # FP32 positions of a box of side 110 (half an ulp 4e-6, one rounding a step)
    assert np.abs(x0 - x3).max() < 2e-4
    assert np.allclose(e0[:, 2:4], e3[:, 2:4], rtol=1e-6)


def test_more_records_than_the_shared_table_build_holds(pkg):
    """Density 4: 370 neighbours an atom in more records than LDS takes, so the
    waves' records are joined in memory (then the kernels for dense systems)."""
    n = 4100
    L = (n / 4.0) ** (1.0 / 3.0)
    x, q = pkg.synth.lattice_positions(n, L, 3), pkg.synth.balanced_charges(n, 3)
    out = []
    for walk in (0, 3):
        sim = pkg.Simulation(n, pkg.SimSpec(duration=0, stepwidth=1e-5, rc=2.5, rc_coul=2.5, skin=0.3, rebuild_every=4,
                                            lo=0.0, hi=L, precision="fp64", energy_every=1, atomsperleaf=5,
                                            resort_every=8, list_walk=walk))
        sim.set_state(x, np.zeros((n, 3)), q)
        sim.run(13)
        out.append((np.array(sim.get_state()[2]), np.array(sim.energies())))
    (f0, e0), (f3, e3) = out
    assert np.array_equal(e0[:, 4], e3[:, 4])
    # 13 steps of FP64 rounding in sums of 370 pair forces
    assert np.abs(f0 - f3).max() < 1e-10 * np.abs(f3).max()
