"""The CSR build of sorted pairs by two splits, at sizes where its tiles,
groups of rows and digits end."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILE = 16384  # entries of a tile of a small input


@pytest.fixture(scope="module")
def split_ctx():
    """A context that builds every sorted input by two splits."""
    from kc_cuda_amd import Context
    mp = pytest.MonkeyPatch()
    mp.setenv("KT_SPLIT_BUILD_MIN", "2")
    c = Context(0)
    mp.undo()
    yield c
    c.close()


def _pairs(kind, n, m):
    rng = np.random.default_rng(m)
    if kind == "hub":  # vertex n - 1 and vertex 0 joined with nearly all others
        ends = np.concatenate([np.column_stack([np.zeros(n - 1, np.int64), np.arange(1, n)]),
                               np.column_stack([np.arange(1, n - 1), np.full(n - 2, n - 1)])])
    else:
        k = rng.choice(n * (n - 1) // 2, m, replace=False) if n < 3000 else None
        if k is not None:  # the k-th pair u < v
            v = ((1 + np.sqrt(1 + 8 * k.astype(np.float64))) / 2).astype(np.int64)
            v -= v * (v - 1) // 2 > k
            v += v * (v + 1) // 2 <= k
            ends = np.column_stack([k - v * (v - 1) // 2, v])
        else:
            lo = n // 5  # empty rows at both ends
            e = rng.integers(lo, n - lo, (2 * m, 2))
            e = e[e[:, 0] != e[:, 1]]
            key = np.unique(np.minimum(e[:, 0], e[:, 1]) * n + np.maximum(e[:, 0], e[:, 1]))
            key = np.sort(rng.choice(key, m, replace=False))
            ends = np.column_stack([key // n, key % n])
    order = np.lexsort((ends[:, 1], ends[:, 0]))
    return ends[order].astype(np.uint32)


@pytest.mark.parametrize("kind,n,m", [
    ("dense", 513, 2), ("dense", 1025, TILE - 1), ("dense", 1536, TILE), ("dense", 2999, TILE + 1),
    ("sparse", 40000, 3 * TILE + 5), ("sparse", 300001, 100000), ("hub", 30000, 0)])
def test_split_build_matches_sorted_rows(split_ctx, kind, n, m):
    pairs = _pairs(kind, n, m)
    split_ctx.solve_pairs(pairs, n)
    off, adj = split_ctx.last_csr(n, 2 * len(pairs))
    p = pairs.astype(np.int64)
    key = np.sort(np.concatenate([p[:, 0] * n + p[:, 1], p[:, 1] * n + p[:, 0]]))
    want = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))])
    np.testing.assert_array_equal(off.astype(np.int64), want)
    rows = np.repeat(np.arange(n, dtype=np.int64), np.diff(want))
    np.testing.assert_array_equal(np.sort(rows * n + adj), key)


@pytest.mark.parametrize("kind,n,m", [
    ("dense", 1025, TILE // 2 - 1), ("dense", 1536, TILE // 2), ("sparse", 40000, TILE + 5), ("hub", 30000, 0)])
def test_split_build_of_shuffled_pairs(split_ctx, kind, n, m):
    """Both entries of every pair are split."""
    pairs = _pairs(kind, n, m)
    pairs = np.ascontiguousarray(pairs[np.random.default_rng(1).permutation(len(pairs))])
    split_ctx.solve_pairs(pairs, n)
    off, adj = split_ctx.last_csr(n, 2 * len(pairs))
    p = pairs.astype(np.int64)
    key = np.sort(np.concatenate([p[:, 0] * n + p[:, 1], p[:, 1] * n + p[:, 0]]))
    want = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))])
    np.testing.assert_array_equal(off.astype(np.int64), want)
    rows = np.repeat(np.arange(n, dtype=np.int64), np.diff(want))
    np.testing.assert_array_equal(np.sort(rows * n + adj), key)
