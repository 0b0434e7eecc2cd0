"""Sorts of up to 8,192 keys by counting each key's predecessors: order and
stability at the edges of its runs of 16 keys and of its range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 15, 16, 17, 1023, 1025, 4096, 8191, 8192, 8193])
@pytest.mark.parametrize("kind", ["ties", "signed", "edges"])
def test_rank_sort_is_stable(pkg, n, kind):
    rng = np.random.default_rng(n)
    if kind == "ties":
        codes = rng.integers(0, max(2, n // 7), n)
    elif kind == "signed":
        codes = rng.integers(-2 ** 31, 2 ** 31, n)
    else:
        codes = rng.choice([-2 ** 31, -1, 0, 2 ** 31 - 1], n)
    codes = codes.astype(np.int32)
    cs, perm = pkg.sortperm(codes)
    ref = np.argsort(codes, kind="stable")
    assert np.array_equal(np.asarray(perm), ref)
    assert np.array_equal(np.asarray(cs), codes[ref])
