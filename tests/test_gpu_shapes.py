"""Sizes at which the kernels change how they split their work: lengths around
the edges of their tiers, remainders, the smallest and largest of a range.
Everything is integer or bit-exact, so results equal the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sess():
    import g500
    s = g500.Session(arena_bytes=8 << 30)
    yield s
    s.close()


@pytest.fixture
def arena(sess):
    m = sess.mark()
    yield sess
    sess.release(m)


def build(arena, n, edges, weights=None):
    edges = np.asarray(edges, np.uint64).reshape(-1, 2)
    if weights is None:
        weights = np.random.default_rng(len(edges)).random(len(edges)).astype(np.float32)
    g = arena.csr(arena.upload_tuples(edges, weights), n)
    import pyoracle
    return g, pyoracle.csr(n, edges, weights)


def two_stars(length):
    """Vertices 0 and 1, both joined to 2 .. length + 1, and to each other: rows of length + 1, a second level of 2."""
    leaves = np.arange(2, length + 2)
    e = [np.stack([np.full(length, c), leaves], 1) for c in (0, 1)] + [np.array([[0, 1]])]
    return length + 2, np.concatenate(e)


@pytest.mark.parametrize("length", [1, 7, 8, 15, 16, 62, 63, 64, 1022, 1023, 1024, 1025, 5000])
def test_depths_of_rows_of_every_tier(arena, oracle, length):
    n, edges = two_stars(length)
    n += 3  # isolated vertices at the end
    g, ref = build(arena, n, edges)
    b = arena.bfs_create(g)
    for root in (0, 2):
        arena.bfs(g, b, root)
        pred = arena.bfs_pred(b)
        trees = [pred.copy() for _ in range(6)]
        trees[1][1] = n - 1          # a centre's parent is no neighbour of it
        trees[2][0 if root else 2] = n + 5
        trees[3][length + 1] = 0     # the last leaf hangs off a centre
        trees[4][[0, 1]] = [1, 0]    # a cycle of the two centres
        trees[5][n - 2] = 1          # an isolated vertex with a parent
        for k, t in enumerate(trees):
            arena.to_device(b.pred, t)
            got = arena.bfs_depth(g, b, root)
            assert np.array_equal(got, oracle.dist_from_pred(ref, t, root)), (length, root, k)


@pytest.mark.parametrize("n", [2, 33, 34, 100, 4099])
def test_depths_of_long_chains(arena, oracle, n):
    order = np.random.default_rng(n).permutation(n)
    g, ref = build(arena, n, np.stack([order[:-1], order[1:]], 1))
    b = arena.bfs_create(g)
    root = int(order[0])
    arena.bfs(g, b, root)
    assert np.array_equal(arena.bfs_depth(g, b, root), oracle.bfs(ref, root)[1])
    pred = arena.bfs_pred(b)
    pred[order[1]] = order[min(2, n - 1)]  # the chain hangs off a cycle (or a loop) next to the root
    arena.to_device(b.pred, pred)
    assert np.array_equal(arena.bfs_depth(g, b, root), oracle.dist_from_pred(ref, pred, root))


# bottom-up levels of the batched BFS: rows below and above the degree that is
# split over the grid (256 on graphs of these sizes), and around the 4096-entry spans
@pytest.mark.parametrize("length", [255, 256, 257, 4095, 4096, 4097, 8192, 20000])
@pytest.mark.parametrize("nroots", [1, 5, 64])
def test_batch_bfs_bottom_up_long_rows(arena, oracle, length, nroots):
    n, edges = two_stars(length)
    n += 7  # a tail of three vertices off the last leaf (the discovery log holds 8n records), four isolated ones
    chain = np.stack([np.arange(n - 8, n - 5), np.arange(n - 7, n - 4)], 1)
    g, ref = build(arena, n, np.concatenate([edges, chain]))
    b = arena.batch_create(g)
    rng = np.random.default_rng(length)
    roots = np.concatenate([[n - 5, 0, 2, n - 1, n - 8], rng.integers(0, n, 59)])[:nroots]
    old = arena.get_param("batch_alpha")
    try:
        arena.set_param("batch_alpha", 1e9)  # every level bottom-up
        arena.batch(g, b, roots)
    finally:
        arena.set_param("batch_alpha", old)
    for i in sorted({0, 1, 2, 3, 4, nroots - 1} & set(range(nroots))):
        assert np.array_equal(arena.batch_depth(g, b, i), oracle.bfs(ref, int(roots[i]))[1]), (length, i)


# edge ranges that end inside tiles and runs of tiles, every remainder of the levels (five at a time),
# and enough edges that some take a rejected number (4 in 10^5)
@pytest.mark.parametrize("scale,start,end", [(1, 0, 32), (2, 3, 61), (4, 0, 257), (6, 255, 1024), (18, 255, 1100001),
                                             (21, 1, 20000001), (24, 2**28 - 9_000_000, 2**28)])
def test_generator_runs_and_remainders(arena, oracle, scale, start, end):
    e, w = arena.tuples_to_host(arena.generate(scale, 16, start=start, end=end))
    eo, wo = oracle.kronecker(scale, 16, start=start, end=end)
    assert np.array_equal(e, eo)
    assert np.array_equal(w.view(np.uint32), wo.view(np.uint32))


def csr_equal(arena, g, ref):
    rs, col, w = arena.csr_to_host(g)
    assert np.array_equal(rs, ref.rowstarts)
    assert np.array_equal(col, ref.column)
    assert np.array_equal(w.view(np.uint32), ref.weights.view(np.uint32))


# tuple lists large enough for the partition: vertex counts around its digit
# splits (two passes up to 2^18, three above), one so sparse that a tile spans
# more buckets than it ranks, a hub with half of all entries, and loops
@pytest.mark.parametrize("n", [3, 255, 1000, 2**18 - 1, 2**18, 2**18 + 1, 700001, 2**22 + 5, 3 * 10**7])
def test_csr_partition(arena, oracle, n):
    rng = np.random.default_rng(n)
    ne = 2**20 + 4097
    e = rng.integers(0, n, (ne, 2))
    if n == 2**18:
        e[: ne // 2, 0] = n - 1
    if n == 1000:
        e[:5000, 1] = e[:5000, 0]
    if n == 3 * 10**7:  # a dense corner and rows far apart
        e[: ne // 2] %= 4096
    g, ref = build(arena, n, e)
    csr_equal(arena, g, ref)


@pytest.mark.parametrize("ne", [2**16 - 1, 2**16])
def test_csr_partition_rejects_endpoints_out_of_range(arena, ne):
    import g500
    e = np.random.default_rng(1).integers(0, 5000, (ne, 2)).astype(np.uint64)
    e[ne // 3, 1] = 5000
    tg = arena.upload_tuples(e, np.ones(ne, np.float32))
    with pytest.raises(g500.LibraryError, match="outside"):
        arena.csr(tg, 5000)


# rows at the edges of the sort's tiers, with evenly spread weights and with
# weights that put many entries, or all, into one bin; with `bulk`, a long row
# more, enough that long rows are sorted in bins
@pytest.mark.parametrize("weights", ["uniform", "equal", "two", "wide", "negative", "infinite"])
@pytest.mark.parametrize("bulk", [0, 150000])
def test_csr_row_sort_tiers(arena, oracle, weights, bulk):
    rng = np.random.default_rng(5)
    lengths = [2, 15, 16, 17, 63, 64, 65, 127, 128, 129, 255, 256, 257, 384, 511, 512, 513, 768, 769, 1025, 4095, 4096,
               4097, 9000] + ([bulk] if bulk else [])
    n = 30000
    e = np.concatenate([np.stack([np.full(d, i), rng.integers(len(lengths), n, d)], 1)
                        for i, d in enumerate(lengths)])
    e = e[rng.permutation(len(e))]
    w = rng.random(len(e)).astype(np.float32)
    if weights == "equal":
        w[:] = 0.25
    elif weights == "two":
        w = np.where(w < 0.5, np.float32(0.1), np.float32(0.9))
    elif weights == "wide":
        w = np.exp(60 * w - 40).astype(np.float32)
    elif weights == "negative":
        w -= np.float32(0.5)
    elif weights == "infinite":
        w[::97] = np.inf
    g, ref = build(arena, n, e, w)
    csr_equal(arena, g, ref)


# the SSSP copy: weights on and next to the steps of the 8-bit hub table, above
# its range and infinite, rows on both sides of a wave, and a graph with few
# entries per vertex in an arena without room for that table
@pytest.mark.parametrize("n,ne,tight", [(40, 300, False), (2000, 30000, False), (9000, 200000, False),
                                        (1 << 20, 3000, True)])
def test_sssp_copy_of_step_weights(arena, oracle, n, ne, tight):
    from test_gpu_pipeline import check_sssp_copy
    rng = np.random.default_rng(ne)
    e = np.minimum(rng.integers(0, n, (ne, 2)), rng.integers(0, n, (ne, 2)) * rng.integers(0, 2, (ne, 2)))
    step = (rng.integers(0, 300, ne) / 127).astype(np.float32)
    w = (step + rng.choice([0.0, 2.0**-10, 2.0**-20, -2.0**-20], ne)).astype(np.float32)
    w = np.where(rng.random(ne) < 0.5, w / 8, w).astype(np.float32)
    w = np.maximum(w, np.float32(0))
    w[::501] = np.inf
    tg = arena.upload_tuples(e, w)
    a, m = arena.ws.gpu_arena, 2 * ne
    saved = a.reserved
    if tight:
        a.reserved = a.used + 176 * n + 24 * m + (9 << 20)
    try:
        g = arena.csr(tg, n)
    finally:
        a.reserved = saved
    check_sssp_copy(arena, g)


# both builds of the batched kernel, and both sides of the line between them
# (entries times roots / 1024 = (1.5 resident roomy blocks)^2: between 18 and 19
# roots here on 256 CUs)
@pytest.mark.parametrize("scale,nroots", [(6, 1), (6, 32), (18, 16), (18, 18), (18, 20), (18, 32)])
def test_batch_sssp_packed_and_roomy(arena, oracle, scale, nroots):
    n = 1 << scale
    g = arena.csr(arena.generate(scale), n)
    ref = oracle.csr(n, *oracle.kronecker(scale))
    roots = np.resize(oracle.roots(ref), nroots).astype(np.uint64)
    sb, s1 = arena.sssp_batch_create(g, 0.05), arena.sssp_create(g, 0.05)
    arena.sssp_batch(g, sb, roots)
    for i, r in enumerate(roots):
        d, p = arena.sssp_batch_result(g, sb, i)
        if i in (0, nroots - 1):
            want = oracle.dijkstra_f32(ref, int(r))[0]
            assert oracle.sssp_check(ref, int(r), d, p) == 0, i
        else:
            arena.sssp(g, s1, int(r))
            want = arena.sssp_result(s1)[0]
        assert np.array_equal(d.view(np.uint32), want.view(np.uint32)), i


# pulled buckets: rows on both sides of a lane's, 16 lanes' and a wave's, with
# ties, infinite weights and scans that end at once or reach the last entry
@pytest.mark.parametrize("length", [1, 3, 4, 5, 31, 62, 63, 64, 65, 127, 510, 511, 512, 513, 3000])
@pytest.mark.parametrize("prune", [0, 1])
def test_sssp_pull_rows_of_every_tier(arena, oracle, length, prune):
    rng = np.random.default_rng(length)
    n, e = two_stars(length)
    e = np.concatenate([e, rng.integers(0, n, (n // 2, 2))]).astype(np.uint64)
    for kind in ("heavy", "mixed", "equal"):
        w = {"heavy": 0.5 + 0.4 * rng.random(len(e)), "mixed": rng.random(len(e)),
             "equal": np.full(len(e), 0.75)}[kind].astype(np.float32)
        if kind == "mixed":
            w[::7] = np.inf
        m = arena.mark()
        saved = {k: arena.get_param(k) for k in ("sssp_pull", "sssp_prune")}
        try:
            arena.set_param("sssp_prune", prune)
            g, ref = build(arena, n, e, w)
            s = arena.sssp_create(g, 0.1)
            for pull in (1e-9, 0.0, 0.3):
                arena.set_param("sssp_pull", pull)
                for root in (0, 2, length + 1):
                    arena.sssp(g, s, root)
                    d, p = arena.sssp_result(s)
                    want, tree = oracle.dijkstra_f32(ref, root)
                    assert np.array_equal(d.view(np.uint32), want.view(np.uint32)), (kind, pull, root)
                    # an infinite entry between a reached and an unreached vertex counts in the oracle's own tree too
                    assert oracle.sssp_check(ref, root, d, p) == oracle.sssp_check(ref, root, want, tree), (kind, root)
        finally:
            for k, x in saved.items():
                arena.set_param(k, x)
            arena.release(m)
