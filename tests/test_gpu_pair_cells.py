"""The lists' passes over cells against the general walks, pair for pair and in
order: the stream-ordered form walks the tree one wave per query group, and
neighbor_traverse follows the ropes of a given tree.  Inputs sit where the
cell passes can go wrong: waves and groups of 16 atoms not filled, pairs at
the radius to the bit, coordinates whose last place is not small against the
radius, crowded cells, more hits than a queue or the LDS holds, an outlier
that stretches the grid (where the call walks the tree), and bad radii."""
import ctypes

import numpy as np
import pytest
from conftest import bruteforce_np, pairs_to_rows, rows_canonical

pytestmark = pytest.mark.gpu


def _points(shape, n, seed):
    rng = np.random.default_rng(seed)
    if shape == "uniform":
        x = rng.random((n, 3)) * (n / 0.8) ** (1 / 3)
    elif shape == "unit":
        x = rng.random((n, 3))
    elif shape == "grid":  # many pairs at s == r * r exactly
        k = int(np.ceil(n ** (1 / 3)))
        x = rng.permutation(np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3))[:n] * 0.5
    elif shape == "line":
        x = np.zeros((n, 3))
        x[:, 0] = rng.random(n) * n / 4
    elif shape == "plane":
        x = rng.random((n, 3)) * [n ** 0.5, 0.0, n ** 0.5]
    elif shape == "point":
        x = np.full((n, 3), 0.25)
    elif shape == "far":  # the last place of 2e4 against r = 1
        x = rng.random((n, 3)) * (n / 0.8) ** (1 / 3) + 2e4
    elif shape == "dense":
        x = rng.random((n, 3)) * 0.5
    else:  # "outlier"
        x = rng.random((n, 3)) * (n / 0.8) ** (1 / 3)
        x[n // 2] = 9e5
    return x.astype(np.float32)


def _general(pkg, x, spec, pred, key):
    """The stream-ordered form's list."""
    ctx, lib = pkg.default_context(), pkg.library()
    d = pkg.DeviceArray.from_host(ctx, x)
    cnt, st = pkg.DeviceArray(ctx, (1,), np.int64), pkg.DeviceArray(ctx, (1,), np.int32)

    def call(out, cap):
        assert lib.nd_leafbuild_traverse_bvh_async(ctx.handle, d.ptr, ctypes.byref(spec.c), pred, key, out, cap,
                                                   cnt.ptr, st.ptr) == 0
        ctx.synchronize()
        assert int(st.to_host()[0]) == 0
        return int(cnt.to_host()[0])

    n = call(None, 0)
    out = pkg.DeviceArray(ctx, (max(n, 1),), pkg.PAIR_DTYPE)
    assert call(out.ptr, n) == n
    return out.to_host(n)


CASES = [
    # shape, n, apl, r
    ("uniform", 2, 1, 1.0), ("uniform", 6, 3, 1.0), ("uniform", 15, 5, 2.0), ("uniform", 16, 4, 2.0),
    ("uniform", 17, 1, 2.0), ("uniform", 1000, 4, 2.8), ("uniform", 4095, 5, 2.8), ("uniform", 4096, 8, 2.8),
    ("uniform", 4160, 64, 1.3), ("uniform", 4160, 65, 1.3), ("uniform", 6000, 2, 1.1), ("uniform", 30003, 3, 1.7),
    ("unit", 4000, 4, 0.05), ("unit", 4000, 1, 0.3), ("unit", 4000, 16, 0.01),
    ("grid", 2000, 4, 1.0), ("grid", 2001, 3, 1.5), ("grid", 2000, 1, 0.5),
    ("line", 1200, 4, 1.0), ("plane", 2000, 2, 1.5), ("point", 96, 4, 0.5), ("point", 96, 1, 1e-3),
    ("far", 3000, 4, 1.0), ("far", 3000, 3, 2e-3), ("dense", 600, 2, 0.7), ("dense", 2200, 1, 0.9),
    ("dense", 1200, 16, 0.4), ("outlier", 4000, 4, 2.0), ("outlier", 12000, 3, 1.0),
    ("uniform", 300, 4, 1e-20), ("uniform", 300, 4, 1e19), ("uniform", 300, 4, 0.0), ("uniform", 300, 4, -1.0),
]


@pytest.mark.parametrize("pred", [0, 1])
@pytest.mark.parametrize("shape,n,apl,r", CASES)
def test_leaf_list_matches_the_walk(pkg, shape, n, apl, r, pred):
    x = _points(shape, n, n + apl)
    spec = pkg.SpheresBVHSpecs(neighbor_distance=r, atom_count=n, atomsperleaf=apl)
    for key in (pkg.MORTON_INTERLEAVE, pkg.MORTON_MASKED):
        want = pairs_to_rows(_general(pkg, x, spec, pred, key))
        out, m = pkg.neighborlist_device(x, spec, pred, key)
        assert np.array_equal(pairs_to_rows(out.to_host(m)) if m else want[:0], want)


@pytest.mark.parametrize("query", [0, 1])
@pytest.mark.parametrize("shape,n,apl,r", [c for c in CASES if c[3] > 0])
def test_point_list_matches_the_ropes(pkg, shape, n, apl, r, query):
    x = _points(shape, n, n + apl)
    spec = pkg.SpheresBVHSpecs(neighbor_distance=r, atom_count=n, atomsperleaf=apl)
    for key in (pkg.MORTON_INTERLEAVE, pkg.MORTON_MASKED):
        got = pkg.build_traverse_bvh(x, spec, key, query)
        nodes, prim, _ = pkg.bvh.tree_export(spec, x)
        want = pkg.neighbor_traverse(nodes, prim, spec, query)
        assert np.array_equal(pairs_to_rows(got), pairs_to_rows(want))


@pytest.mark.parametrize("pred", [0, 1])
@pytest.mark.parametrize("shape,n,r", [("uniform", 15, 2.0), ("uniform", 17, 2.0), ("uniform", 4097, 2.8),
                                       ("grid", 2000, 1.0), ("far", 3000, 1.0), ("point", 700, 0.5),
                                       ("dense", 1500, 0.9), ("dense", 1500, 1e3), ("line", 1200, 1e-22),
                                       ("uniform", 800, 1e20)])
def test_cell_list_is_the_definition(pkg, shape, n, r, pred):
    x = _points(shape, n, n)
    got = rows_canonical(pairs_to_rows(pkg.cell_neighborlist(x, r, pred)))
    assert np.array_equal(got, bruteforce_np(x, r, pred))


def test_too_small_a_buffer_is_left_alone(pkg):
    """Nothing is written when the list does not fit, and the tree is there."""
    n = 5000
    x = _points("uniform", n, 9)
    ctx, lib = pkg.default_context(), pkg.library()
    d = pkg.DeviceArray.from_host(ctx, x)
    spec = pkg.SpheresBVHSpecs(neighbor_distance=2.5, atom_count=n, atomsperleaf=4)
    sentinel = np.full(64, -7, np.int32)
    out = pkg.DeviceArray.from_host(ctx, sentinel)
    count = ctypes.c_int64(0)
    for call in (lambda: lib.nd_leafbuild_traverse_bvh(ctx.handle, d.ptr, ctypes.byref(spec.c), 0, 1, out.ptr, 16,
                                                       ctypes.byref(count)),
                 lambda: lib.nd_build_traverse_bvh(ctx.handle, d.ptr, ctypes.byref(spec.c), 0, 1, out.ptr, 16,
                                                   ctypes.byref(count))):
        assert call() == -3 and count.value > 16
        assert np.array_equal(out.to_host(), sentinel)
        assert len(pkg.bvh.tree_export(spec, x)[0]) == 2 * spec.leaves_count - 1
