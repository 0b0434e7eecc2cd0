"""Adjoint: lists that outgrow the room made for the first one.  The pass runs on
with rows cut short and is repeated, so what it found after that is not this
system's."""
import numpy as np
import pytest
import torch
from scipy.spatial import cKDTree

pytestmark = pytest.mark.gpu


def _inwards(pkg, n, density, rate):
    """A lattice whose atoms all move to its centre."""
    L = pkg.synth.box_side(n, density)
    x = pkg.synth.lattice_positions(n, L, 3)
    return x, -rate * (x - L / 2), pkg.synth.balanced_charges(n, 3), L ** 3


@pytest.mark.parametrize("every,rebuild", [(40, 10), (10, 5), (40, 1)])
def test_gradients_where_later_lists_have_longer_rows(pkg, O, every, rebuild):
    n, steps, skin = 512, 40, 1.5
    x, v, q, V = _inwards(pkg, n, 0.3, 5.0)
    target = np.linspace(0.0, 1.5, 20)
    reach = 2.65 + skin
    assert max(map(len, cKDTree(x).query_ball_point(x, reach))) - 1 <= 96  # the first list fits
    adj = pkg.Adjoint(n, steps, dt=0.002, precision="fp64", checkpoint_every=every, rebuild_every=rebuild, nbins=20,
                      rdf_rmax=2.5, rdf_h=0.15, volume=V, skin=skin)
    op = O.Adj64Params(eps=1.0, sigma=1.0, rc=2.5, k_coul=1.0, rc_coul=2.5, dt=0.002, rdf_rmax=2.5, rdf_h=0.15,
                       volume=V, nbins=20, nsteps=steps)
    L_o, g_o, dx_o, dv_o, dq_o, dp_o = O.adj64_run(x, v, q, op, target=target, grads=True)
    for _ in range(2):
        L, g = adj.forward(x, v, q, target)
        xT = adj.final_state()[0]
        gr = adj.backward()
        assert abs(L - L_o) < 1e-9 * abs(L_o)
        assert np.allclose(g, g_o, rtol=1e-9, atol=1e-12)
        for name, want in (("dx0", dx_o), ("dv0", dv_o), ("dq", dq_o), ("deps", dp_o[0]), ("dsigma", dp_o[1])):
            assert np.abs(gr[name] - want).max() <= 1e-8 * max(1.0, np.abs(want).max()), name
    assert max(map(len, cKDTree(xT).query_ball_point(xT, reach))) - 1 > 96  # the last does not
    adj.close()


def test_rows_are_sized_for_this_system(pkg):
    """The memory taken follows the system's own rows (at most four times the
    longest), not those of the pass without room, in which atoms gather: 1,480 MB
    where the longest row is 275 and five lists of rows of 960 take 630."""
    n, every = 32768, 10
    x, v, q, V = _inwards(pkg, n, 0.6, 20.0)
    kw = dict(dt=0.002, precision="fp64", checkpoint_every=40, rebuild_every=every, nbins=20, rdf_rmax=2.5, rdf_h=0.1,
              volume=V)
    longest = 0
    for steps in (0, 10, 20, 30, 40):  # positions of each list, from a pass that ends there
        xT = x
        if steps:
            adj = pkg.Adjoint(n, steps, **kw)
            adj.forward(x, v, q)
            xT = adj.final_state()[0]
            adj.close()
        longest = max(longest, cKDTree(xT).query_ball_point(xT, 2.9001, return_length=True).max() - 1)
    assert longest > 96
    adj = pkg.Adjoint(n, 40, **kw)
    before = torch.cuda.mem_get_info()[0]
    adj.forward(x, v, q)
    taken = before - torch.cuda.mem_get_info()[0]
    adj.close()
    # five lists (four windows and the final positions), 4 bytes an entry; the allocator's granularity
    assert taken <= 5 * 4 * n * (4 * longest + 8) + (64 << 20)
