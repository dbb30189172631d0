"""Options and arenas at the ends of their ranges: what a knob's extreme values
do, the smallest arena that a construction takes, inputs that leave a split of
the work with few pieces. Everything is integer or bit-exact."""
import numpy as np
import pytest

from test_gpu_shapes import arena, build, csr_equal, sess, two_stars  # noqa: F401 (fixtures)

pytestmark = pytest.mark.gpu


# the vertices that a bottom-up level splits over the grid are those above the
# knob's degree, whatever the graph's size; only the default leaves the degree
# to the library
@pytest.mark.parametrize("heavy", [1, 200, 300, 1024, 4096, 5000, 1 << 30])
def test_batch_heavy_degree_is_the_split_degree(arena, oracle, heavy):
    n, edges = two_stars(5000)
    rng = np.random.default_rng(heavy)
    mid = np.stack([np.repeat(np.arange(2, 12), 400), rng.integers(2, n, 4000)], 1)  # ten rows of 400 and more
    g, ref = build(arena, n, np.concatenate([edges, mid]))
    degree = np.diff(ref.rowstarts.astype(np.int64))
    b = arena.batch_create(g)
    default = arena.get_param("batch_heavy_degree")
    assert default == 1 << 20
    roots = np.array([2, n - 1, 0, 7], np.uint64)
    old = arena.get_param("batch_alpha")
    try:
        arena.set_param("batch_alpha", 1e9)  # every level bottom-up
        arena.set_param("batch_heavy_degree", heavy)
        arena.to_device(b.hub_lengths, np.zeros(3 * n, np.uint32))
        arena.batch(g, b, roots)
    finally:
        arena.set_param("batch_alpha", old)
        arena.set_param("batch_heavy_degree", default)
    listed = arena.to_host(b.hub_lengths, 3 * n, np.uint32)[2 * n:]
    assert np.array_equal(np.sort(listed[listed > 0]), np.sort(degree[degree > heavy]))
    for i, r in enumerate(roots):
        assert np.array_equal(arena.batch_depth(g, b, i), oracle.bfs(ref, int(r))[1]), i
