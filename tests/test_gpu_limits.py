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


def hub_row(weights):
    """A vertex with an entry to random others for each of the weights."""
    n = 1 << 20
    other = np.random.default_rng(9).integers(1, n, len(weights))
    return n, np.stack([np.zeros(len(weights), np.int64), other], 1), weights.astype(np.float32)


def rows_ms(arena, tg, n):
    """Device time of the rows alone (no copies), the least of five."""
    old = arena.get_param("relabel")
    arena.set_param("relabel", 0)
    try:
        ms = []
        for _ in range(5):
            m = arena.mark()
            arena.csr(tg, n)
            ms.append(arena.lib.g500_last_run_ms())
            arena.release(m)
        return min(ms)
    finally:
        arena.set_param("relabel", old)


# One long row whose weights are not evenly spread: over-full bins, which blocks
# sort. With squared uniform weights the first of 2605 bins holds 10^6 / sqrt(2605)
# = 19600 entries (one block's radix sort, 40 ns an entry: 0.8 ms) and some 360 more
# of 513 to 8000 are over-full; spread over the chip those cost no more than the
# evenly spread row's whole construction (0.5 ms) again. So about 3.6 times that,
# 6 with a margin; 13 when the blocks are as many as the long rows.
def test_over_full_bins_of_one_row_are_sorted_side_by_side(arena, oracle):
    u = np.random.default_rng(10).random(10**6)
    n, e, w = hub_row(u * u)
    g, ref = build(arena, n, e, w)
    csr_equal(arena, g, ref)
    even, skewed = (rows_ms(arena, arena.upload_tuples(e, x.astype(np.float32)), n) for x in (u, w))
    print(f"[over-full bins] evenly spread {even:.3f} ms, squared {skewed:.3f} ms", flush=True)
    assert skewed < 6 * even


# One long row of equal weights is one bin, which one block sorts. That costs as
# much per entry as a row of 131000 entries, which is short enough to be sorted as
# it lies, and the construction's other costs grow slower than the entries: at most
# the ratio of the entries, with 5 % for the clock. 9.0 to 7.6 when the bin is
# copied by one wave first; 70 to 30.5 when a row with more bins than are counted in
# LDS makes a global atomic per entry.
@pytest.mark.parametrize("entries", [10**6, 4 * 10**6])
def test_a_row_of_equal_weights_costs_a_sort_as_it_lies(arena, oracle, entries):
    ms = {}
    for k in (131000, entries):
        n, e, w = hub_row(np.full(k, 0.25))
        g, ref = build(arena, n, e, w)
        csr_equal(arena, g, ref)
        ms[k] = rows_ms(arena, arena.upload_tuples(e, w), n)
    print(f"[equal weights] {ms}", flush=True)
    assert ms[entries] < 1.05 * entries / 131000 * ms[131000]


# rows around one and two rounds of 8192 bins counted at a time (384 entries a
# bin), alone and with a second row in the same span, evenly spread or not
@pytest.mark.parametrize("entries", [384 * 8192, 384 * 8192 + 1, 2 * 384 * 8192 + 5000])
def test_rows_of_more_bins_than_one_round(arena, oracle, entries):
    rng = np.random.default_rng(entries)
    u = rng.random(entries)
    u[::3] *= u[::3]  # some over-full bins at the light end
    n, e, w = hub_row(u)
    second = np.stack([np.ones(600, np.int64), rng.integers(2, n, 600)], 1)  # its chunks follow the hub's
    e, w = np.concatenate([e, second]), np.concatenate([w, rng.random(600).astype(np.float32)])
    g, ref = build(arena, n, e, w)
    csr_equal(arena, g, ref)


def round256(x):
    return (x + 255) // 256 * 256


# A construction of rows alone needs, beside the CSR, 24 bytes a vertex for the sort's
# lists and 8 an entry of rows above 4096 for its scratch, each array rounded to 256
# bytes. Many entries per vertex (lists by entries would need more than that), rows of
# every tier; with hubs, whose scratch is most of the room.
@pytest.mark.parametrize("hubs", [0, 3])
def test_rows_in_the_smallest_arena(arena, oracle, hubs):
    rng = np.random.default_rng(hubs)
    n = 3000
    deg = np.concatenate([rng.integers(600, 1500, 1700), rng.integers(0, 40, 600), rng.integers(40, 500, 695),
                          np.full(hubs, 60000), np.full(5 - hubs, 1)])
    e = np.stack([np.repeat(np.arange(n), deg), rng.integers(0, n, deg.sum())], 1)
    if not hubs:  # every row at most 4096 entries
        assert np.bincount(e.ravel(), minlength=n).max() <= 4096
    w = rng.random(len(e)).astype(np.float32)
    tg = arena.upload_tuples(e, w)
    ref = oracle.csr(n, e.astype(np.uint64), w)
    degree = np.diff(ref.rowstarts.astype(np.int64))
    m, huge = int(degree.sum()), int(degree[degree > 4096].sum())
    assert (huge > 0) == (hubs > 0)
    need = round256(8 * (n + 1)) + 2 * round256(4 * m)
    need += 4 * round256(4 * n) + round256(8 * n) + 256 + 2 * round256(4 * huge)
    a, saved, old = arena.ws.gpu_arena, arena.ws.gpu_arena.reserved, arena.get_param("relabel")
    arena.set_param("relabel", 0)
    a.reserved = round256(a.used) + need
    try:
        g = arena.csr(tg, n)
        mark = a.used
    finally:
        a.reserved = saved
        arena.set_param("relabel", old)
    assert g.notisolated == int((degree > 0).sum())
    assert mark <= g.weights + 4 * m - a.base + 255  # the scratch is released
    csr_equal(arena, g, ref)


# The SSSP copy is built where 8 bytes an entry and 144 a vertex and 8 MiB are
# free beside the traversal copy, also where the entries are so many (40000 a
# vertex) that the bits of the kept ones, 1/7 byte each with their offsets, are
# more than the hub table.
def test_sssp_copy_of_a_dense_graph_in_little_room(arena):
    scale = 11
    n = 1 << scale
    tg = arena.generate(scale, 20000)
    a, saved, m0 = arena.ws.gpu_arena, arena.ws.gpu_arena.reserved, arena.mark()
    kept = []  # entries kept per original vertex
    for tight in (False, True):
        arena.release(m0)
        if tight:
            m = int(g.nlocaledges)
            rows = round256(8 * (n + 1)) + 2 * round256(4 * m)
            traversal = 2 * round256(4 * n) + round256(8 * (n + 1)) + 2 * round256(4 * m)
            a.reserved = round256(a.used) + rows + traversal + 256 + 8 * (n + 1) + 8 * m + 136 * n + (8 << 20)
        try:
            g = arena.csr(tg, n)
        finally:
            a.reserved = saved
        assert g.rowstarts_s, tight
        rs = arena.to_host(g.rowstarts_s, n + 1, np.uint64).astype(np.int64)
        kept.append(np.diff(rs)[arena.to_host(g.perm, n, np.uint32)])
    assert np.array_equal(*kept) and kept[0].sum() < m
    s = arena.sssp_create(g, 0.1)
    root = int(arena.roots(g)[0])
    arena.sssp(g, s, root)
    assert arena.sssp_check(g, s.dist, s.pred, root) == 0


# Persistent kernels on every block that the device holds, with small blocks: the
# grid barrier's largest member counts. Grids follow the work (entries / 512 or
# 256, times roots), and S24's fills the device at these shapes: plain BFS
# sqrt(5.3e8 / 512) x 512 / 128 = 4060 blocks wanted of 128 threads where 3072 are
# resident, 2030 of 256 where 1536 are; the others hold fewer.
@pytest.fixture(scope="module")
def s24():
    import g500
    s = g500.Session(arena_bytes=64 << 30)
    g = s.csr(s.generate(24), 1 << 24)
    yield s, g, s.roots(g)[:6]
    s.close()


KNOBS = ("bfs_block", "sssp_block", "batch_bfs_block", "batch_sssp_block")


def traversals(s, g, roots):
    """Depths and distances by each of the four kernels."""
    m, out, some = s.mark(), [], (0, len(roots) - 1)
    b, p = s.bfs_create(g), s.sssp_create(g, 0.1)
    for i in some:
        s.bfs(g, b, roots[i])
        assert s.bfs_validate(g, b, roots[i]) == (True, 0)
        out.append(s.bfs_depth(g, b, roots[i]))
        s.sssp(g, p, roots[i])
        assert s.sssp_check(g, p.dist, p.pred, roots[i]) == 0
        out.append(s.sssp_result(p)[0].view(np.uint32))
    s.release(m)
    bb = s.batch_create(g)
    s.batch(g, bb, roots)
    out += [s.batch_depth(g, bb, i) for i in some]
    s.release(m)
    sb = s.sssp_batch_create(g, 0.05)
    s.sssp_batch(g, sb, roots)
    out += [s.sssp_batch_result(g, sb, i)[0].view(np.uint32) for i in some]
    s.release(m)
    return out


def test_small_blocks_on_the_whole_device(s24):
    s, g, roots = s24
    old = {k: s.get_param(k) for k in KNOBS}
    want = traversals(s, g, roots)
    for i in (0, 2):  # the batched kernels agree with the plain ones
        assert np.array_equal(want[i], want[4 + i // 2]) and np.array_equal(want[i + 1], want[6 + i // 2])
    try:
        for block in (128, 256):
            for k in KNOBS:
                s.set_param(k, block)
            for k, (x, y) in enumerate(zip(want, traversals(s, g, roots))):
                assert np.array_equal(x, y), (block, k)
    finally:
        for k, v in old.items():
            s.set_param(k, v)


# A launch's blocks follow the vertices as well as the entries: with an entry per 40
# vertices a launch is a pass over per-vertex arrays, about as much as a copy of 32
# bytes a vertex (the labels, probes, stamps and row records that SSSP touches; the
# batched BFS touches less). Both within twice that; 4 and 2.2 times with the 24 and
# 32 blocks that the entries alone ask for.
def test_few_entries_over_many_vertices(arena, oracle):
    n = 8 * 10**6
    e = np.random.default_rng(3).integers(0, n, (10**5, 2))
    g, ref = build(arena, n, e)
    root = int(e[0, 0])
    m = arena.mark()
    size = 32 * n
    src = arena.lib._worker_arena_push_array(arena.ws, size, 1, 256, None)
    dst = arena.lib._worker_arena_push_array(arena.ws, size, 1, 256, None)

    def best(run):
        run()
        return min(run() for _ in range(5))

    def copy():
        arena.lib.g500_copy_device(dst, src, size)
        return arena.lib.g500_last_run_ms()

    ms = {"copy": best(copy)}
    arena.release(m)
    s, b = arena.sssp_create(g), arena.batch_create(g)
    ms["sssp"] = best(lambda: arena.sssp(g, s, root))
    ms["batch"] = best(lambda: arena.batch(g, b, np.array([root], np.uint64)))
    print(f"[few entries] {ms}", flush=True)
    want = oracle.dijkstra_f32(ref, root)[0]
    assert np.array_equal(arena.sssp_result(s)[0].view(np.uint32), want.view(np.uint32))
    assert np.array_equal(arena.batch_depth(g, b, 0), oracle.bfs(ref, root)[1])
    assert max(ms["sssp"], ms["batch"]) < 2 * ms["copy"]


# The validation's pieces: rows around the length that a whole wave walks, alone and
# behind each other, and around the pieces of 128 rows and entries of small graphs
@pytest.mark.parametrize("length", [1, 63, 125, 126, 127, 128, 129, 255, 256, 257, 5000])
def test_validation_counts_in_pieces(arena, oracle, length):
    n, edges = two_stars(length)
    n += 200  # isolated vertices at the end
    g, ref = build(arena, n, edges)
    b = arena.bfs_create(g)
    for root in (0, length + 1):
        arena.bfs(g, b, root)
        pred = arena.bfs_pred(b)
        trees = [pred.copy() for _ in range(6)]
        trees[1][1] = n - 1          # a centre's parent is no neighbour of it
        trees[2][0 if root else 2] = n + 5
        trees[3][length + 1] = length + 1
        trees[4][[0, 1]] = [1, 0]    # a cycle of the two centres
        trees[5][n - 2] = 1          # an isolated vertex with a parent
        for k, t in enumerate(trees):
            arena.to_device(b.pred, t)
            ok, errors = arena.bfs_validate(g, b, root)
            assert errors == oracle.bfs_validate(ref, t, root) and ok == (errors == 0), (root, k)


# 64 hubs with following ids, and the same graph with its ids shuffled: the rows of the
# hubs are cut into pieces either way. 17 times when one wave walks all of them.
def test_validation_of_hubs_that_follow_each_other(arena):
    import time
    rng = np.random.default_rng(2)
    n, ne = 500064, 3 * 10**6
    e = np.stack([rng.integers(0, 64, ne), 64 + rng.integers(0, n - 64, ne)], 1)
    ms = []
    for ids in (np.arange(n), rng.permutation(n)):
        m = arena.mark()
        g = arena.csr(arena.upload_tuples(ids[e], rng.random(ne).astype(np.float32)), n)
        b = arena.bfs_create(g)
        root = int(ids[0])
        arena.bfs(g, b, root)
        times = []
        for _ in range(6):
            t0 = time.perf_counter()
            assert arena.bfs_validate(g, b, root) == (True, 0)
            times.append(time.perf_counter() - t0)
        ms.append(1e3 * min(times))
        arena.release(m)
    print(f"[hub validate] ids in order {ms[0]:.3f} ms, shuffled {ms[1]:.3f} ms", flush=True)
    assert ms[0] < 3 * ms[1]


# Tuples that lie near the ones before them are placed through cursors, whose atomics
# and writes then share lines; in shuffled order the partition is the faster. 0.48 of
# the shuffled order's time on a path of 1e7 vertices, 0.81 when both are partitioned.
def test_tuples_in_order_are_not_partitioned(arena, oracle):
    n = 10**7
    e = np.stack([np.arange(n - 1), np.arange(1, n)], 1)
    rng = np.random.default_rng(4)
    w = rng.random(n - 1).astype(np.float32)
    ms = []
    for order in (np.arange(n - 1), rng.permutation(n - 1)):
        m = arena.mark()
        tg = arena.upload_tuples(e[order], w[order])
        ms.append(rows_ms(arena, tg, n))
        old = arena.get_param("relabel")
        arena.set_param("relabel", 0)
        g = arena.csr(tg, n)
        arena.set_param("relabel", old)
        if not len(ms) - 1:
            rows = arena.csr_to_host(g)
        else:
            assert all(np.array_equal(x, y) for x, y in zip(rows, arena.csr_to_host(g)))
        arena.release(m)
    print(f"[tuples ms] in order {ms[0]:.3f}, shuffled {ms[1]:.3f}", flush=True)
    assert ms[0] < 0.65 * ms[1]


# the sample that decides it: lists around its block of 1024 tuples and its eight blocks,
# near ones, and near ones with every third on the vertex before
@pytest.mark.parametrize("ne", [2**18, 2**18 + 1, 2**19 + 1023, 2**20 + 8192])
@pytest.mark.parametrize("kind", ["near", "on", "descending", "far"])
def test_orders_of_tuples(arena, oracle, ne, kind):
    i = np.arange(ne)
    e = {"near": np.stack([i, i + 7], 1), "on": np.stack([i // 3, i + 1], 1),
         "descending": np.stack([ne - i, ne - i + 16], 1), "far": np.stack([i * 17 % ne, i], 1)}[kind]
    g, ref = build(arena, ne + 20, e)
    csr_equal(arena, g, ref)


# The SSSP copy of a graph without hubs: its rows are judged by the exact hub table,
# 128 bytes a vertex written and read (one copy's time) and about as much again for the
# passes over rows and entries. 2.15 copies on a path of 1e7 vertices; 2.8 with the 8-bit
# table, which pays only where many rows reach a hub.
def test_sssp_copy_of_a_graph_without_hubs(arena):
    n = 10**7
    e = np.stack([np.arange(n - 1), np.arange(1, n)], 1)
    tg = arena.upload_tuples(e, np.random.default_rng(5).random(n - 1).astype(np.float32))

    def best(run):
        ms = []
        for _ in range(6):
            m = arena.mark()
            run()
            ms.append(arena.lib.g500_last_run_ms())
            arena.release(m)
        return min(ms)

    old = arena.get_param("sssp_prune")
    try:
        ms = {}
        for prune in (0, 1):
            arena.set_param("sssp_prune", prune)
            ms[prune] = best(lambda: arena.csr(tg, n))
    finally:
        arena.set_param("sssp_prune", old)
    size = 128 * n
    src, dst = (arena.lib._worker_arena_push_array(arena.ws, size, 1, 256, None) for _ in range(2))
    ms["copy"] = best(lambda: arena.lib.g500_copy_device(dst, src, size))
    print(f"[no hubs ms] {ms}", flush=True)
    assert ms[1] - ms[0] < 2.5 * ms["copy"]
