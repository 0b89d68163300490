"""Solves while the device has little memory left: triangle lists are an
option that a core does without, and the room they took goes to other buffers."""
import ctypes
from contextlib import contextmanager

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL("libamdhip64.so").hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@contextmanager
def _all_but(ctx, left):
    """Holds the device's free memory except `left` bytes."""
    from kc_cuda_amd import native_library
    held = []
    try:
        while (more := min(_free_bytes() - left, 32 << 30)) > 0:
            p = ctypes.c_void_p()
            assert native_library().kt_malloc(ctx._h, more, ctypes.byref(p)) == 0
            held.append(p)
        yield
    finally:
        for p in held:
            assert native_library().kt_free(ctx._h, p) == 0


def _clique(n):
    u, v = np.triu_indices(n, 1)
    return np.column_stack([u, v]).astype(np.uint32)


def _near_clique(n):
    """A clique of n - 1 and a vertex joined with half of it: supports differ, so triangles are listed."""
    return np.concatenate([_clique(n - 1), np.column_stack([np.arange(n // 2), np.full(n // 2, n - 1)]).astype(np.uint32)])


@pytest.fixture
def sparse_ctx():
    from kc_cuda_amd import Context
    with Context(0) as c:
        c.tune(core="sparse")
        yield c


def test_lists_that_cannot_be_allocated(sparse_ctx):
    """600 vertices: 862 MB of lists for 180 k edges, with 256 MB left."""
    sparse_ctx.solve_pairs(_clique(8), 8)
    with _all_but(sparse_ctx, 256 << 20):
        t = sparse_ctx.solve_pairs(_near_clique(601), 601), sparse_ctx.trussness()
    again = sparse_ctx.solve_pairs(_near_clique(601), 601), sparse_ctx.trussness()
    for r, rows in (t, again):
        assert (r.kmax, r.truss_edges) == (600, 600 * 599 // 2)
        np.testing.assert_array_equal(np.unique(rows[:, 2], return_counts=True), [[301, 600], [300, 600 * 599 // 2]])


def test_room_of_old_lists_goes_to_other_buffers(sparse_ctx):
    """4 M edges take some 300 MB, of which 128 MB are left beside the lists
    of an earlier core."""
    n = 601
    r = sparse_ctx.solve_pairs(_near_clique(n), n)
    assert r.truss_edges == (n - 1) * (n - 2) // 2
    sparse_ctx.trussness()  # lists its triangles
    rng = np.random.default_rng(1)
    m = 4_000_000
    u = np.sort(rng.integers(0, 1 << 20, m)).astype(np.uint32)
    pairs = np.column_stack([u, (1 << 20) + np.arange(m, dtype=np.uint32) % (1 << 19)])
    pairs = np.concatenate([_clique(30), pairs])
    pairs = np.unique(pairs, axis=0)
    held = sparse_ctx.to_device(pairs)
    with _all_but(sparse_ctx, 128 << 20):
        r = sparse_ctx.solve_device(held, len(pairs), 3 << 19)
    held.free()
    assert (r.kmax, r.truss_edges) == (30, 435)
