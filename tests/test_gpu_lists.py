"""Truss levels over triangle lists against the oracle, and against the rows
that a core whose triangles do not fit the budget is peeled with."""
import numpy as np
import pytest

from conftest import canon_pairs
from graphs import closed_forms, random_graph
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _graphs():
    from kc_cuda_amd import gen
    out = [(name, np.asarray(p, np.uint32).reshape(-1, 2), n) for name, p, n, _, _ in closed_forms()]
    for seed, (n, p, cl) in enumerate([(60, 0.4, (9,)), (300, 0.06, (12, 9)), (700, 0.05, ())]):
        out.append((f"er{seed}", random_graph(n, p, seed, cliques=cl), n))
    out.append(("rmat11", *gen.rmat(11, 8, 0.57, 0.19, 0.19, True, 9, 3)))
    return out


@pytest.fixture(scope="module", params=["lists", "rows"])
def sparse_ctx(request):
    """A context that keeps every core in sorted rows; "rows": no room for lists."""
    from kc_cuda_amd import Context
    mp = pytest.MonkeyPatch()
    if request.param == "rows":
        mp.setenv("KT_LIST_BUDGET_MB", "0")
    c = Context(0)
    mp.undo()
    c.tune(core="sparse")
    yield c
    c.close()


def test_sparse_cores_match_oracle(sparse_ctx):
    for name, pairs, n in _graphs():
        print(f"[gpu] {name} m={len(pairs)}", flush=True)
        ref = O.solve_pairs(pairs, n, want_edges=True)
        r = sparse_ctx.solve_pairs(pairs, n)
        assert (r.k_hat, r.kmax, r.truss_edges) == (ref.k_hat, ref.kmax, ref.truss_edges), name
        np.testing.assert_array_equal(sparse_ctx.truss_edges(), canon_pairs(ref.truss), err_msg=name)
        t = O.trussness(pairs)
        want = np.array(sorted((u, v, k) for (u, v), k in t.items() if k >= 3), dtype=np.uint32).reshape(-1, 3)
        np.testing.assert_array_equal(sparse_ctx.trussness(), want, err_msg=name)


@pytest.mark.parametrize("scale,lanes", [(14, 8), (14, 64), (15, 0)])
def test_lists_equal_rows(ctx, sparse_ctx, scale, lanes):
    """Frontiers from one edge to hundreds of thousands (several edges a wave,
    several waves an edge), live lists rewritten on the way: every trussness."""
    from kc_cuda_amd import gen
    pairs, n = gen.rmat(scale, 16, 0.57, 0.19, 0.19, True, 20, 4)
    sparse_ctx.tune(core="sparse", count_lanes=lanes)
    try:
        r = sparse_ctx.solve_pairs(pairs, n)
        got = sparse_ctx.trussness()
    finally:
        sparse_ctx.tune(core="sparse")
    ref = ctx.solve_pairs(pairs, n)
    assert (r.kmax, r.truss_edges, r.k_hat) == (ref.kmax, ref.truss_edges, ref.k_hat)
    np.testing.assert_array_equal(got, ctx.trussness())


@pytest.fixture(scope="module", params=["eid_matrix", "prefix_counts"])
def dense_ctx(request):
    """A context that keeps every core in bit-matrix rows; "prefix_counts": no
    room for the matrix of edge ids."""
    from kc_cuda_amd import Context
    mp = pytest.MonkeyPatch()
    if request.param == "prefix_counts":
        mp.setenv("KT_EIDM_BUDGET_MB", "0")
    c = Context(0)
    mp.undo()
    c.tune(core="dense")
    yield c
    c.close()


# row words: one, two, the support count's lane steps (128 and 256), the last
@pytest.mark.parametrize("n", [64, 65, 2048, 8191, 16385, 65536])
def test_dense_rows_equal_lists(dense_ctx, n):
    """The whole decomposition over bit-matrix rows: walks, dropped frontiers
    cleared edge by edge or by rebuilding the rows, recounts, the stops where
    the host shrinks the matrix or leaves it."""
    from kc_cuda_amd import Context
    rng = np.random.default_rng(n)
    m = min(n * (n - 1) // 4, 60_000)
    e = rng.integers(0, n, (m, 2))
    k = min(n, 300)  # a dense corner: sparse edges go first, in drops
    c = rng.integers(0, k, (25 * k, 2))
    e = np.concatenate([e, c, np.column_stack([np.arange(n), (np.arange(n) + 1) % n]),
                        np.column_stack([np.arange(n), (np.arange(n) + 2) % n])])
    pairs = np.unique(canon_pairs(e[e[:, 0] != e[:, 1]].astype(np.uint32)), axis=0)
    r = dense_ctx.solve_pairs(pairs, n)
    got = dense_ctx.trussness()
    with Context(0) as other:
        other.tune(core="sparse")
        ref = other.solve_pairs(pairs, n)
        want = other.trussness()
    assert (r.kmax, r.truss_edges, r.k_hat) == (ref.kmax, ref.truss_edges, ref.k_hat)
    np.testing.assert_array_equal(got, want)


# a row: one word, whole runs of words and one more, more slots than one pass
# over a row takes
@pytest.mark.parametrize("n", [3, 64, 1024, 1025, 2050])
def test_dense_views_of_cliques(dense_ctx, n):
    """A clique hung with triangles: the level's rows hold vertices outside
    the core, ranks run against ids."""
    u, v = np.triu_indices(n, 1)
    t = np.arange(n)
    pairs = np.concatenate([np.column_stack([u, v]), np.column_stack([t, n + t])]).astype(np.uint32)
    pairs = canon_pairs((2 * n - 1 - pairs).astype(np.uint32))
    r = dense_ctx.solve_pairs(pairs, 2 * n)
    assert (r.kmax, r.truss_edges, r.max_core) == (n, n * (n - 1) // 2, n - 1)
    got = dense_ctx.truss_edges()
    assert (got >= n).all() and len(np.unique(got[:, 0].astype(np.uint64) * (2 * n) + got[:, 1])) == len(got)


# rows one bit past a word, one short of it, whole chunks of eight words, and
# squares of row blocks
@pytest.mark.parametrize("n,p", [(1601, 0.6), (1727, 0.6), (2048, 0.4), (6000, 0.1)])
def test_counts_by_pairs_equal_rows(dense_ctx, n, p):
    """Cores whose supports are counted by all pairs of rows on the matrix
    cores, at first and after every dropped frontier: every trussness."""
    from kc_cuda_amd import Context
    rng = np.random.default_rng(n)
    pairs = np.argwhere(np.triu(rng.random((n, n), dtype=np.float32) < p, 1)).astype(np.uint32)
    r = dense_ctx.solve_pairs(pairs, n)
    got = dense_ctx.trussness()
    assert r.recounts > 0
    with Context(0) as other:
        other.tune(core="sparse")
        ref = other.solve_pairs(pairs, n)
        want = other.trussness()
    assert (r.kmax, r.truss_edges, r.k_hat) == (ref.kmax, ref.truss_edges, ref.k_hat)
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("seed", [1, 2])
def test_one_sided_lines_equal_rows(dense_ctx, seed):
    """Lines that list some edges in one direction only, as many each way (two
    copies of a graph, the other half of the lines left out in each), solve as
    on a core of sorted rows."""
    from kc_cuda_amd import Context
    n = 130
    e = np.asarray(random_graph(n, 0.4, seed, cliques=(12,)), np.uint32).reshape(-1, 2)
    cut = np.random.default_rng(seed).random(len(e)) < 0.1
    both = np.concatenate([e, e[:, ::-1]])
    a = np.concatenate([both[:len(e)], both[len(e):][~cut]])
    b = np.concatenate([both[:len(e)][~cut], both[len(e):]]) + n
    lines = np.concatenate([a, b]).astype(np.uint32)
    lines = lines[np.lexsort((lines[:, 0], lines[:, 1]))]
    xs, ys = np.ascontiguousarray(lines[:, 0]), np.ascontiguousarray(lines[:, 1])
    r = dense_ctx.solve_lines(xs, ys, 2 * n)
    with Context(0) as other:
        other.tune(core="sparse")
        ref = other.solve_lines(xs, ys, 2 * n)
        want = other.truss_edges()
    assert (r.kmax, r.truss_edges, r.k_hat) == (ref.kmax, ref.truss_edges, ref.k_hat)
    np.testing.assert_array_equal(dense_ctx.truss_edges(), want)


@pytest.mark.parametrize("by_edge", [False, True])
def test_rows_that_repeat_a_neighbour_are_not_listed(by_edge):
    """Pairs given more than once: the two support counts find different
    triangles on such rows, so they are peeled by rows, whatever the budget."""
    from kc_cuda_amd import Context
    rng = np.random.default_rng(7)
    once = np.argwhere(np.triu(rng.random((80, 80)) < 0.4, 1))
    pairs = np.concatenate([once, once[rng.random(len(once)) < 0.3]]).astype(np.uint32)
    mp = pytest.MonkeyPatch()
    mp.setenv("KT_LIST_BUDGET_MB", "0")
    with Context(0) as rows:
        mp.undo()
        rows.tune(core="sparse", force_edge_count=by_edge)
        want = rows.solve_pairs(pairs, 80)
        want_t = rows.trussness()
    with Context(0) as lists:
        lists.tune(core="sparse", force_edge_count=by_edge)
        got = lists.solve_pairs(pairs, 80)
        assert (got.kmax, got.truss_edges, got.k_hat) == (want.kmax, want.truss_edges, want.k_hat)
        np.testing.assert_array_equal(lists.trussness(), want_t)


def test_repeated_pairs_on_dense_cores(dense_ctx):
    """Every copy of an edge has its support counted, at first and after
    dropped frontiers, whatever the last solve left behind."""
    n = 1300  # counted by all pairs of rows, were no pair repeated
    u, v = np.triu_indices(n, 1)
    once = np.column_stack([u, v]).astype(np.uint32)
    twice = np.repeat(once, 2, axis=0)
    for _ in range(2):
        r = dense_ctx.solve_pairs(twice, n)
        assert (r.kmax, r.truss_edges) == (n, len(twice))
        np.testing.assert_array_equal(dense_ctx.truss_edges(), twice)
        rng = np.random.default_rng(3)  # other supports in the same buffers
        dense_ctx.solve_pairs(once[rng.random(len(once)) < 0.6], n)
    # sparse edges on a repeated clique: they go first, in drops
    tail = np.argwhere(np.triu(np.random.default_rng(4).random((3000, 3000), dtype=np.float32) < 0.05, 1)) + n // 2
    pairs = np.concatenate([twice, tail[tail[:, 1] >= n].astype(np.uint32)])
    got = []
    for other in (once, tail.astype(np.uint32)):
        dense_ctx.solve_pairs(other, n // 2 + 3000)
        r = dense_ctx.solve_pairs(pairs, n // 2 + 3000)
        got.append((r.kmax, r.truss_edges, dense_ctx.truss_edges()))
    assert got[0][:2] == got[1][:2] == (n, len(twice))
    np.testing.assert_array_equal(got[0][2], twice)
    np.testing.assert_array_equal(got[1][2], twice)


@pytest.mark.parametrize("side", [3, 40, 90])
def test_cores_without_triangles(sparse_ctx, side):
    """Nothing is listed; the levels end in their first look."""
    i = np.arange(side * side).reshape(side, side)
    pairs = canon_pairs(np.concatenate([np.column_stack([i[:, :-1].ravel(), i[:, 1:].ravel()]),
                                        np.column_stack([i[:-1].ravel(), i[1:].ravel()])]).astype(np.uint32))
    for _ in range(2):
        r = sparse_ctx.solve_pairs(pairs, side * side)
        assert (r.max_core, r.kmax, r.truss_edges) == (2, 0, 0)
        assert len(sparse_ctx.truss_edges()) == 0 and len(sparse_ctx.trussness()) == 0
        k5 = np.array([(a, b) for a in range(5) for b in range(a + 1, 5)], dtype=np.uint32)
        assert sparse_ctx.solve_pairs(k5, 5).kmax == 5


@pytest.mark.parametrize("kind,size", [("cliques", 5), ("cliques", 40), ("wheel", 4), ("wheel", 5), ("wheel", 900),
                                       ("wheel_and_tail", 30)])
def test_searches_that_walk_no_frontier(sparse_ctx, kind, size):
    """Equal supports, or a first level that ends the search: nothing is
    listed; and next to them searches that do walk."""
    if kind == "cliques":
        u, v = np.triu_indices(size, 1)
        pairs, n = np.concatenate([np.column_stack([u, v]) + i * size for i in range(20)]), 20 * size
    else:
        rim = np.arange(1, size + 1)
        pairs, n = np.concatenate([np.column_stack([np.zeros(size, int), rim]), np.column_stack([rim, rim % size + 1])]), size + 1
        if kind == "wheel_and_tail":  # a square: supports below the first level
            pairs, n = np.concatenate([pairs, [[0, n], [n, n + 1], [n + 1, 1]]]), n + 2
    pairs = np.unique(canon_pairs(pairs.astype(np.uint32)), axis=0)
    ref = O.solve_pairs(pairs, n, want_edges=True)
    r = sparse_ctx.solve_pairs(pairs, n)
    assert (r.k_hat, r.kmax, r.truss_edges) == (ref.k_hat, ref.kmax, ref.truss_edges)
    np.testing.assert_array_equal(sparse_ctx.truss_edges(), canon_pairs(ref.truss))
    t = O.trussness(pairs)
    want = np.array(sorted((u, v, k) for (u, v), k in t.items() if k >= 3), dtype=np.uint32).reshape(-1, 3)
    np.testing.assert_array_equal(sparse_ctx.trussness(), want)
