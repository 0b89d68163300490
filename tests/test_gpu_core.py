"""The max-core search by core numbers: every branch of its sweeps (one
workgroup; estimates in LDS or in memory; rows of a lane group, a wave, a
workgroup in registers and longer) and the peel that takes over when they do
not converge, against the oracle."""
import numpy as np
import pytest

from conftest import canon_pairs
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _hubs(n, degrees, m, clique, seed):
    """m random edges, a clique, and hubs joined to the first `degree` other vertices."""
    rng = np.random.default_rng(seed)
    e = [rng.integers(0, n, (m, 2))]
    vs = rng.choice(n, clique, replace=False)
    e.append(np.array([(a, b) for i, a in enumerate(vs) for b in vs[i + 1:]]).reshape(-1, 2))
    for h, d in enumerate(degrees):
        e.append(np.column_stack([np.full(d, h), (h + 1 + np.arange(d)) % n]))
    e = np.concatenate(e)
    return np.unique(canon_pairs(e[e[:, 0] != e[:, 1]].astype(np.uint32)), axis=0)


def _lollipop(path, clique):
    """A clique with a path hanging off it."""
    e = [(a, b) for a in range(clique) for b in range(a + 1, clique)]
    e += [(clique - 1 + i, clique + i) for i in range(path)]
    return np.array(e, dtype=np.uint32)


CASES = {
    # one workgroup, up to its limits of 4,096 vertices and 8,192 row slots, and past them
    "tiny": (40, [], 100, 6), "one_wg": (4096, [900], 3000, 9), "past_n": (4097, [900], 3000, 9),
    "past_slots": (900, [], 4200, 9),
    # LDS estimates: rows past a lane group, a wave (4,096) and the registers of a workgroup (16,384)
    "lds_rows": (30_000, [300, 1200, 4096, 4097, 16_384, 16_385, 29_000], 60_000, 20),
    "lds_dense": (3_000, [2_999, 2_500], 200_000, 60),
    "lds_last_n": (65_536, [17_000], 40_000, 12),
    # estimates in memory: one workgroup of 256 holds 4,096 row entries in registers
    "memory": (65_537, [300, 1200, 4096, 4097, 20_000], 100_000, 14),
}


@pytest.mark.parametrize("name", CASES)
def test_max_core_of_every_row_length(ctx, name):
    n, hubs, m, clique = CASES[name]
    pairs = _hubs(n, hubs, m, clique, len(name))
    ref = O.solve_pairs(pairs, n, want_edges=True)
    r = ctx.solve_pairs(pairs, n)
    assert (r.max_core, r.k_hat, r.kmax, r.truss_edges) == (ref.max_core, ref.k_hat, ref.kmax, ref.truss_edges)
    np.testing.assert_array_equal(ctx.truss_edges(), canon_pairs(ref.truss))


@pytest.mark.parametrize("path", [1, 511, 513, 1200, 5000])
def test_cores_that_unravel_along_a_path(ctx, path):
    """Each sweep moves the end of the path by one vertex; past the sweeps'
    limit the peel takes over."""
    pairs = _lollipop(path, 7)
    r = ctx.solve_pairs(pairs, 7 + path)
    assert (r.max_core, r.kmax, r.truss_edges) == (6, 7, 21)


@pytest.mark.parametrize("down", [False, True])
@pytest.mark.parametrize("vertex", ["cascade", "rounds", "auto"])
def test_lines_in_one_direction_only(ctx, vertex, down):
    """Rows that do not mirror each other, searched by peels with a cut at 275
    of 2,000 vertices: the same answer twice, and the right one for the next
    graph. The peels' degrees do not size such rows, and sweeps of core numbers,
    which mark a vertex's own row, do not find their fixpoint."""
    from kc_cuda_amd import Context
    rng = np.random.default_rng(6)
    e = np.argwhere(np.triu(rng.random((2000, 2000), dtype=np.float32) < 0.012, 1))
    x, y = (e[:, 1], e[:, 0]) if down else (e[:, 0], e[:, 1])
    order = np.lexsort((x, y))
    xs, ys = x[order].astype(np.uint32), y[order].astype(np.uint32)
    pairs = e.astype(np.uint32)
    ref = O.solve_pairs(pairs, 2000)
    with Context(0) as c:
        c.tune(vertex=vertex)
        one = c.solve_lines(xs, ys, 2000)
        two = c.solve_lines(xs, ys, 2000)
        assert (one.max_core, one.k_hat, one.kmax, one.truss_edges) == (two.max_core, two.k_hat, two.kmax, two.truss_edges)
        r = c.solve_pairs(pairs, 2000)
        assert (r.max_core, r.kmax, r.truss_edges) == (ref.max_core, ref.kmax, ref.truss_edges)


@pytest.mark.parametrize("copies", [4000, 65534, 65535, 65536, 70000])
def test_cores_of_repeated_pairs_beyond_16_bits(ctx, copies):
    """Two vertices joined many times: a core as large as the count of copies."""
    r = ctx.solve_pairs(np.tile(np.array([[3, 9]], np.uint32), (copies, 1)), 12)
    assert (r.max_core, r.kmax, r.truss_edges) == (copies, 0, 0)


def _grid(side, diagonals):
    i = np.arange(side * side).reshape(side, side)
    e = [np.column_stack([i[:, :-1].ravel(), i[:, 1:].ravel()]), np.column_stack([i[:-1].ravel(), i[1:].ravel()])]
    if diagonals:
        e.append(np.column_stack([i[:-1, :-1].ravel(), i[1:, 1:].ravel()]))
    return canon_pairs(np.concatenate(e).astype(np.uint32)), side * side


def _ladder_into_expander(columns, n):
    """A ladder, broken at one end, that leads into a random graph: every
    vertex has three neighbours, so the 3-core unravels along the ladder and
    then all over the graph at once."""
    rng = np.random.default_rng(n)
    ring = np.arange(n)
    match = rng.permutation(n).reshape(-1, 2)  # a ring and a matching
    e = np.concatenate([np.column_stack([ring, (ring + 1) % n])[:-1], match])  # the ring is cut between n - 1 and 0
    u, v = n + np.arange(columns), n + columns + np.arange(columns)
    e = np.concatenate([e, np.column_stack([u[:-1], u[1:]]), np.column_stack([v[:-1], v[1:]]), np.column_stack([u, v]),
                        [[0, u[-1]], [n - 1, v[-1]]]])
    return np.unique(canon_pairs(e.astype(np.uint32)), axis=0), n + 2 * columns


def _star_and_tail(leaves, path):
    """A star on the end of a path that leads out of a ring with a chord: the
    ring is the 2-core."""
    ring = 104
    i = np.arange(ring)
    walk = ring - 1 + np.arange(path + 1)
    hub = int(walk[-1])
    e = np.concatenate([np.column_stack([i, (i + 1) % ring]), [[0, 2]], np.column_stack([walk[:-1], walk[1:]]),
                        np.column_stack([np.full(leaves, hub), hub + 1 + np.arange(leaves)])])
    return canon_pairs(e.astype(np.uint32)), hub + 1 + leaves


LONG = {
    # one workgroup from the start, from the first sweeps on, from later ones on; peel with bounds
    "grid_20": lambda: _grid(20, False), "mesh_40": lambda: _grid(40, True), "grid_70": lambda: _grid(70, False),
    "mesh_150": lambda: _grid(150, True), "grid_256": lambda: _grid(256, False), "grid_257": lambda: _grid(257, False),
    "grid_640": lambda: _grid(640, False), "mesh_560": lambda: _grid(560, True),
    "path_4096": lambda: (_lollipop(4089, 7), 4096), "path_65536": lambda: (_lollipop(65_529, 7), 65_536),
    # long rows beside the path: the peel goes on from the estimates
    "star_150": lambda: _star_and_tail(150, 9000), "star_9000": lambda: _star_and_tail(9000, 12_000),
    "star_20000": lambda: _star_and_tail(20_000, 60_000),
    # more vertices due at once than one workgroup lists
    "expander": lambda: _ladder_into_expander(300, 60_000),
}


@pytest.mark.parametrize("name", LONG)
def test_cores_that_unravel_over_many_sweeps(ctx, name):
    pairs, n = LONG[name]()
    print(f"[gpu] {name} m={len(pairs)}", flush=True)
    ref = O.solve_pairs(pairs, n, want_edges=True)
    r = ctx.solve_pairs(pairs, n)
    assert (r.max_core, r.k_hat, r.kmax, r.truss_edges) == (ref.max_core, ref.k_hat, ref.kmax, ref.truss_edges)
    np.testing.assert_array_equal(ctx.truss_edges(), canon_pairs(ref.truss))


@pytest.mark.parametrize("path", [300, 5000, 70_000])
def test_second_core_from_bounds(ctx, path):
    """A max core without triangles, known before the path that hangs off it has
    unravelled: the 2-core of the second pass is peeled from upper bounds."""
    k = 10
    side = np.array([(a, k + b) for a in range(k) for b in range(k)])
    walk = 2 * k - 1 + np.arange(path + 1)
    end = int(walk[-1])
    e = np.concatenate([side, np.column_stack([walk[:-1], walk[1:]]), [[end, end + 1], [end, end + 2], [end + 1, end + 2]],
                        [[end + 2, end + 3]]])  # a triangle, and a spike on it
    e = np.concatenate([e, np.column_stack([np.full(path, end + 3), end + 4 + np.arange(path)])[:1],
                        np.column_stack([end + 4 + np.arange(path - 1), end + 5 + np.arange(path - 1)])])
    n = end + 4 + path
    r = ctx.solve_pairs(canon_pairs(e.astype(np.uint32)), n)
    assert (r.max_core, r.kmax, r.truss_edges) == (k, 3, 3)
    np.testing.assert_array_equal(ctx.truss_edges(), [[end, end + 1], [end, end + 2], [end + 1, end + 2]])


@pytest.mark.parametrize("kept,m", [(300_000, 2_200_000), (540_000, 2_300_000)])
def test_pruned_and_cut_again(ctx, kept, m):
    """A filtered cut of 2^22 row slots and more, pruned with the bitmap of its
    vertices in LDS (up to 524,288 of them) or in memory, and, where enough of
    its vertices hang by fewer than k neighbours, cut a second time."""
    rng = np.random.default_rng(kept)
    n = 4 * kept + 4096
    hubs = 48  # a clique: the h-index is at least 48, the filter's k 4 or so
    core = kept // 2  # joined at random among themselves; the others have a star's centre and two more
    e = [rng.integers(hubs, core, (m, 2))]
    leaf = np.arange(core, kept)
    e.append(np.column_stack([leaf, rng.integers(hubs, core, len(leaf))]))
    e += [np.column_stack([leaf, kept + (leaf * 3 + d) % (n - kept)]) for d in range(5)]
    u, v = np.triu_indices(hubs, 1)
    e.append(np.column_stack([u, v]))
    e.append(np.column_stack([np.arange(hubs), hubs + np.arange(hubs)]))
    e = np.concatenate(e)
    pairs = np.unique(canon_pairs(e[e[:, 0] != e[:, 1]].astype(np.uint32)), axis=0)
    print(f"[gpu] {len(pairs)} edges", flush=True)
    ref = O.solve_pairs(pairs, n, want_edges=True)
    r = ctx.solve_pairs(pairs, n)
    assert (r.max_core, r.k_hat, r.kmax, r.truss_edges) == (ref.max_core, ref.k_hat, ref.kmax, ref.truss_edges)
    np.testing.assert_array_equal(ctx.truss_edges(), canon_pairs(ref.truss))


def test_bounds_of_the_whole_graph_after_filters_without_a_core(ctx):
    """Stars raise the degree h-index, whose filters leave no core; the path
    keeps the whole graph's sweeps from converging, so the peel starts from its
    estimates."""
    stars, leaves, path, clique = 120, 140, 150_000, 7
    base = clique + path  # after the clique with its tail
    centre = base + np.arange(stars) * (leaves + 1)
    e = [_lollipop(path, clique).astype(np.int64),
         np.column_stack([np.repeat(centre, leaves), (centre[:, None] + 1 + np.arange(leaves)).ravel()]),
         np.column_stack([centre[:-1], centre[1:]])]
    pairs = canon_pairs(np.concatenate(e).astype(np.uint32))
    r = ctx.solve_pairs(pairs, int(pairs.max()) + 1)
    assert (r.max_core, r.kmax, r.truss_edges) == (6, 7, 21)
    np.testing.assert_array_equal(ctx.truss_edges(), _lollipop(0, clique))
