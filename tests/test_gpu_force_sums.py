"""Pair-list forces: the workgroups' LDS sums against FP64, and the same bits
in every list order (the sums are integers, so order and grouping cannot
matter; a list in random order names more atoms per workgroup than its table
holds, which takes the overflow to memory)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def coulomb64(x, q, pi, pj, n):
    """FP64 Coulomb forces of FP32 inputs, the sum of the pairs' |f| per atom, the energy."""
    x, q = x.astype(np.float64), q.astype(np.float64)
    d = x[pi] - x[pj]
    r = np.sqrt((d * d).sum(1))
    s = q[pi] * q[pj] / r ** 3
    f, a = np.zeros((n, 3)), np.zeros((n, 3))
    for c in range(3):
        np.add.at(f[:, c], pi, s * d[:, c])
        np.add.at(f[:, c], pj, -s * d[:, c])
        for k in (pi, pj):
            np.add.at(a[:, c], k, np.abs(s) * r)
    return f, a, (q[pi] * q[pj] / r).sum(), np.abs(q[pi] * q[pj] / r).sum()


# sizes around a thread per pair, a run per workgroup, and more atoms in a
# workgroup's run than the table has slots
@pytest.mark.parametrize("n,npairs", [(2, 1), (40, 63), (500, 1023), (500, 1024), (500, 1025), (30000, 262143),
                                      (30000, 1200001)])
def test_sums_match_fp64_in_every_order(pkg, n, npairs):
    rng = np.random.default_rng(n + npairs)
    L = pkg.synth.box_side(n)
    x = pkg.synth.lattice_positions(n, L, 3).astype(np.float32)
    q = rng.uniform(-1.0, 1.0, n).astype(np.float32)
    pi = rng.integers(0, n, npairs).astype(np.int32)
    pj = ((pi + rng.integers(1, n, npairs)) % n).astype(np.int32)
    ref, size, e_ref, e_size = coulomb64(x, q, pi, pj, n)
    got = []
    for order in (np.arange(npairs), np.argsort(pi, kind="stable"), rng.permutation(npairs)):
        p = np.zeros(npairs, pkg.PAIR_DTYPE)
        p["i"], p["j"] = pi[order], pj[order]
        f = np.zeros((n, 3), np.float32)
        e = pkg.force_coulomb_(f, p, q, x, k=1.0, rc=1e6)
        # per pair at most 16 FP32 roundings; 2^-32 per pair of fixed point; one final rounding
        tol = 16 * U * size + 2.0 ** -32 * (1 + np.bincount(np.r_[pi, pj], minlength=n)[:, None]) + U * np.abs(ref)
        assert (np.abs(f - ref) <= tol).all()
        assert abs(e - e_ref) <= 16 * U * e_size
        got.append(f)
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
