"""Adjoint lists of systems that a grid over their box serves badly: clusters far
apart and atoms far out.  Above 1,200 tests an atom the cells of lines take over."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _droplets(pkg, n, parts, place):
    """parts droplets of n / parts atoms, droplet k around place(k)."""
    m = n // parts
    L = pkg.synth.box_side(m)
    x = np.concatenate([pkg.synth.lattice_positions(m, L, 3 + k) - L / 2 + place(k) for k in range(parts)])
    return x, pkg.synth.gaussian_velocities(n, 1.0, 3), pkg.synth.balanced_charges(n, 3)


# two droplets of 1,300 on a diagonal, on a line, around 0 (cells of either sign);
# one droplet and atoms in every direction up to 1e30 out; a droplet and a vapour
@pytest.mark.parametrize("shape", ["diagonal", "line", "negative", "outliers", "vapour"])
@pytest.mark.parametrize("steps,every,rebuild", [(7, 3, 3), (4, 4, 1)])
def test_gradients_of_far_clusters_match_the_oracle(pkg, O, shape, steps, every, rebuild):
    n = 2600
    if shape in ("diagonal", "line", "negative"):
        step = {"diagonal": [700.0, 700.0, 700.0], "line": [9e3, 0.0, 0.0], "negative": [-800.0, 300.0, -500.0]}[shape]
        x, v, q = _droplets(pkg, n, 2, lambda k: np.array(step) * k)
    else:
        x, v, q = _droplets(pkg, n, 1, lambda k: 0.0)
        rng = np.random.default_rng(5)
        if shape == "outliers":
            x[::200] = rng.normal(size=(13, 3)) * 10.0 ** rng.uniform(3, 30, (13, 1))
            v[::200] = 0.0
        else:
            x[::4] = rng.uniform(-400.0, 400.0, (n // 4, 3))
    V = n / 0.8
    target = np.linspace(0.0, 1.5, 20)
    adj = pkg.Adjoint(n, steps, dt=0.002, eps=1.02, sigma=0.98, precision="fp64", checkpoint_every=every,
                      rebuild_every=rebuild, nbins=20, rdf_rmax=2.5, rdf_h=0.15, volume=V)
    op = O.Adj64Params(eps=1.02, sigma=0.98, rc=2.5, k_coul=1.0, rc_coul=2.5, dt=0.002, rdf_rmax=2.5, rdf_h=0.15,
                       volume=V, nbins=20, nsteps=steps)
    L_o, g_o, dx_o, dv_o, dq_o, dp_o = O.adj64_run(x, v, q, op, target=target, grads=True)
    L, g = adj.forward(x, v, q, target)
    gr = adj.backward()
    adj.close()
    assert abs(L - L_o) < 1e-9 * abs(L_o)
    assert np.allclose(g, g_o, rtol=1e-9, atol=1e-12)
    for name, want in (("dx0", dx_o), ("dv0", dv_o), ("dq", dq_o), ("deps", dp_o[0]), ("dsigma", dp_o[1])):
        assert np.abs(gr[name] - want).max() <= 1e-8 * max(1.0, np.abs(want).max()), name


@pytest.mark.parametrize("shape", ["droplets", "outlier"])
def test_distance_does_not_cost(pkg, shape):
    """The same pairs, farther apart: 24 ms against 2.0 with the cells of a box,
    2.2 with lines.  Three times allows for noise."""
    n, steps = 262144, 10
    took = []
    for far in (100.0, 1000.0):
        x, v, q = _droplets(pkg, n, 2, lambda k: np.full(3, far * k if shape == "droplets" else 100.0 * k))
        if shape == "outlier":
            x[7] = 100.0 * far
        adj = pkg.Adjoint(n, steps, dt=0.001, precision="fp64", checkpoint_every=50, rebuild_every=10, nbins=20,
                          rdf_rmax=2.5, rdf_h=0.1, volume=n / 0.8)
        times = []
        for _ in range(4):
            t = time.perf_counter()
            adj.forward(x, v, q)
            times.append(time.perf_counter() - t)
        adj.close()
        took.append(min(times))
    assert took[1] < 3.0 * took[0], took
