"""The adjoint's segments, windows and orders: horizons that end inside a window
or a segment, one window per segment, windows of one step, segments recomputed
from their checkpoints, and more windows than rows are kept for."""
import numpy as np
import pytest
from test_gpu_adjoint import _system

pytestmark = pytest.mark.gpu


# n, steps, checkpoint_every, rebuild_every
@pytest.mark.parametrize("n,steps,every,rebuild", [(48, 1, 50, 10), (48, 10, 10, 10), (48, 11, 10, 10), (48, 37, 20, 5),
                                                   (100, 20, 10, 1), (64, 30, 15, 15), (8, 12, 6, 3),
                                                   (516, 9, 100, 50)])
def test_gradients_match_the_oracle(pkg, O, n, steps, every, rebuild):
    x, v, q, V = _system(n, 7)
    q = q * 1.1
    target = np.linspace(0.0, 1.5, 20)
    adj = pkg.Adjoint(n, steps, dt=0.002, eps=1.02, sigma=0.98, precision="fp64", checkpoint_every=every,
                      rebuild_every=rebuild, nbins=20, rdf_rmax=2.5, rdf_h=0.15, volume=V)
    op = O.Adj64Params(eps=1.02, sigma=0.98, rc=2.5, k_coul=1.0, rc_coul=2.5, dt=0.002, rdf_rmax=2.5, rdf_h=0.15,
                       volume=V, nbins=20, nsteps=steps)
    L_o, g_o, dx_o, dv_o, dq_o, dp_o = O.adj64_run(x, v, q, op, target=target, grads=True)
    for _ in range(2):  # a second call on the same buffers
        L, g = adj.forward(x, v, q, target)
        gr = adj.backward()
        assert abs(L - L_o) < 1e-9 * abs(L_o)
        assert np.allclose(g, g_o, rtol=1e-9, atol=1e-12)
        for name, want in (("dx0", dx_o), ("dv0", dv_o), ("dq", dq_o), ("deps", dp_o[0]), ("dsigma", dp_o[1])):
            assert np.abs(gr[name] - want).max() <= 1e-8 * max(1.0, np.abs(want).max()), name
    adj.close()


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_segment_length_does_not_change_the_gradients(pkg, precision):
    """One segment of 60 one-step windows (more rows than are kept at this
    size: the sweep lists the windows past them again) against segments of 12
    (recomputed from checkpoints, every window's rows kept).  Positions are the
    same to the bit; only the order of FP64 sums differs."""
    n, steps = 200000, 60
    L = pkg.synth.box_side(n)
    x = pkg.synth.lattice_positions(n, L, 5)
    v = pkg.synth.gaussian_velocities(n, 1.0, 5)
    q = pkg.synth.balanced_charges(n, 5)
    target = np.linspace(0.0, 1.5, 50)
    got = []
    for every in (60, 12):
        adj = pkg.Adjoint(n, steps, dt=0.001, precision=precision, checkpoint_every=every, rebuild_every=1, nbins=50,
                          rdf_rmax=2.5, rdf_h=0.1, volume=L ** 3)
        loss, _ = adj.forward(x, v, q, target)
        state = adj.final_state()
        got.append((state, loss, adj.backward()))
        adj.close()
    (sa, la, a), (sb, lb, b) = got
    assert np.array_equal(sa[0], sb[0]) and np.array_equal(sa[1], sb[1])
    assert abs(la - lb) <= 1e-12 * abs(lb)
    for k in ("dx0", "dv0", "dq", "deps", "dsigma"):
        assert np.linalg.norm(np.asarray(a[k]) - b[k]) <= 1e-11 * np.linalg.norm(b[k]), k
