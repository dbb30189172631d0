"""The work that programs have this library do, as cases to be timed.

A case is one call (or one short chain of calls) of the C-ABI through its
Python binding, on inputs that a seed fixes: Kronecker graphs from the
library's own generator with a user seed, or uniform random graphs of a
caller's own. Kinds:

  generate   generate_kronecker_range of an edge range
  construct  oned_graph_from_tuple_graph: the CSR and the copies it carries
  bfs        one root: clear, run, depths from the parent tree; with
             "validate", the Graph500 rules too, as the runner does per root
  sssp       one root: clear, run
  bfs_batch  up to 64 roots in one launch, then every root's depths
  sssp_batch up to 32 roots in one launch, with or without bucket offsets

Parent arrays are left out of the outputs: any parent that achieves the depth
or distance is a right answer and the order of atomics picks one. The BFS
depths are derived from the whole parent array, so they stand for it.

Device memory comes from one arena per state; the arena is a torch tensor, so
that outputs are views of it and it is freed with the state.
"""
import ctypes as C
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "cuda-graph-traversal_amd"))
import g500  # noqa: E402


def listed():
    return [
        # a rank's slice of an edge list: start and end inside 256-edge tiles
        {"name": "generate-s24-slice", "kind": "generate", "scale": 24, "edgefactor": 16, "start": 100_003,
         "end": 250_000_007},
        # a small graph built on demand (interactive use, tests): launches and host waits count
        {"name": "construct-s13-ef5", "kind": "construct", "graph": "kronecker", "scale": 13, "edgefactor": 5},
        # kernel 1 of Graph500 at a size of the serving tier
        {"name": "construct-s23", "kind": "construct", "graph": "kronecker", "scale": 23, "edgefactor": 16},
        # a query on a small resident graph: latency
        {"name": "bfs-s12", "kind": "bfs", "graph": "kronecker", "scale": 12, "edgefactor": 16, "validate": False},
        # a caller's own graph, no hubs, an odd vertex count, validated as the runner validates
        {"name": "bfs-uniform-700001", "kind": "bfs", "graph": "uniform", "vertices": 700_001, "edgefactor": 11,
         "validate": True},
        # the benchmark's graph
        {"name": "bfs-s26", "kind": "bfs", "graph": "kronecker", "scale": 26, "edgefactor": 16, "validate": False},
        # a query on a small resident graph, the reference's delta
        {"name": "sssp-s12", "kind": "sssp", "graph": "kronecker", "scale": 12, "edgefactor": 16, "delta": 0.1},
        # an ordinary graph with an odd edge factor
        {"name": "sssp-s19-ef9", "kind": "sssp", "graph": "kronecker", "scale": 19, "edgefactor": 9, "delta": 0.1},
        # the benchmark's graph at the delta its tuner picks
        {"name": "sssp-s26", "kind": "sssp", "graph": "kronecker", "scale": 26, "edgefactor": 16, "delta": 0.05},
        # 64 roots, depths of every one
        {"name": "bfs-batch-s21x64", "kind": "bfs_batch", "graph": "kronecker", "scale": 21, "edgefactor": 16,
         "roots": 64},
        # what a serving slot launches for a few requests on a small graph
        {"name": "sssp-batch-s16x7", "kind": "sssp_batch", "graph": "kronecker", "scale": 16, "edgefactor": 16,
         "roots": 7, "delta": 0.05, "offsets": False},
        # a full launch with bucket offsets
        {"name": "sssp-batch-s22x32", "kind": "sssp_batch", "graph": "kronecker", "scale": 22, "edgefactor": 16,
         "roots": 32, "delta": 0.05, "offsets": True},
    ]


def draw(rng):
    kind = rng.choice(["generate", "construct", "bfs", "sssp", "bfs_batch", "sssp_batch"])
    if kind == "generate":
        scale = rng.randint(10, 24)
        total = 16 << scale
        count = int(min(total, math.exp(rng.uniform(math.log(1000), math.log(250_000_000)))))
        start = rng.randint(0, total - count)
        return {"kind": kind, "scale": scale, "edgefactor": 16, "start": start, "end": start + count}
    top = {"construct": 22, "bfs": 24, "sssp": 24, "bfs_batch": 20, "sssp_batch": 20}[kind]
    case = {"kind": kind}
    if kind in ("construct", "bfs", "sssp") and rng.random() < 0.3:
        case.update(graph="uniform", vertices=int(math.exp(rng.uniform(math.log(1000), math.log(4_000_000)))))
    else:
        case.update(graph="kronecker", scale=rng.randint(10, top))
    case["edgefactor"] = rng.randint(3, 20)
    if kind == "bfs":
        case["validate"] = rng.random() < 0.3
    elif kind == "sssp":
        case["delta"] = rng.choice([0.05, 0.1, 0.25])
    elif kind == "bfs_batch":
        case["roots"] = rng.randint(2, 64)
    elif kind == "sssp_batch":
        case.update(roots=rng.randint(2, 32), delta=rng.choice([0.025, 0.05, 0.1]), offsets=rng.random() < 0.5)
    return case


def _size(case):
    """(vertices, tuples) of a case's graph."""
    n = case["vertices"] if case.get("graph") == "uniform" else 1 << case["scale"]
    return n, case["end"] - case["start"] if case["kind"] == "generate" else n * case["edgefactor"]


def work(case):
    n, ne = _size(case)
    m = 2 * ne  # directed entries
    kind = case["kind"]
    if kind == "generate":
        return {"bytes": 20 * ne, "flops": 0}
    if kind == "construct":
        return {"bytes": 20 * ne + 8 * m + 8 * n, "flops": 0}
    rows = 4 * m + 8 * n
    if kind == "bfs":
        return {"bytes": rows + 16 * n, "flops": 0}
    if kind == "bfs_batch":
        return {"bytes": rows + 8 * n * case["roots"], "flops": 0}
    return {"bytes": rows + 4 * m + 12 * n * case.get("roots", 1), "flops": m * case.get("roots", 1)}


# ------------------------------------------------------------------ states
_worker = None


class Device(g500.Session):
    """A binding session whose device arena is a torch tensor of its own."""

    def __init__(self, nbytes):
        global _worker
        if _worker is None:  # one worker per process; every state brings its arena
            _worker = g500.Session(1 << 20)
        self.lib = _worker.lib
        self.mem = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()  # the library has a stream of its own
        self.ws = g500.WorkerState.from_buffer_copy(_worker.ws)
        self.ws.gpu_arena = g500.Arena(nbytes, 0, self.mem.data_ptr())

    def view(self, ptr, shape, dtype):
        at = int(ptr) - self.mem.data_ptr()
        size = math.prod(shape) * dtype.itemsize
        return self.mem[at:at + size].view(dtype).view(shape)


def _seeds(seed):
    return (int(seed) % 1_000_003) + 2, (int(seed) // 1_000_003) + 3


def _uniform(case, seed):
    """Edges and weights of a uniform random graph."""
    n, ne = _size(case)
    gen = torch.Generator("cuda").manual_seed(int(seed))
    edges = torch.randint(0, n, (ne, 2), generator=gen, device="cuda")
    return edges, torch.rand(ne, generator=gen, device="cuda")


def _no_loop(a, b, n):
    return torch.where(a == b, (b + 1) % n, b)


def _tuples(dev, case, seed):
    n, ne = _size(case)
    if case["graph"] == "kronecker":
        return dev.generate(case["scale"], case["edgefactor"], *_seeds(seed))
    edges, weights = _uniform(case, seed)
    tg = g500.TupleGraph()
    tg.edges_size = tg.max_edges_size = tg.nglobaledges = ne
    count = g500.u64()
    tg.edges = dev.lib._worker_arena_push_array(C.byref(dev.ws), ne, 16, 16, C.byref(count))
    tg.weights = dev.lib._worker_arena_push_array(C.byref(dev.ws), ne, 4, 4, C.byref(count))
    dev.view(tg.edges, (ne, 2), torch.int64).copy_(edges)
    dev.view(tg.weights, (ne,), torch.float32).copy_(weights)
    torch.cuda.synchronize()
    return tg


def _graph_bytes(n, ne):
    """Arena room of a construction: the CSR, its two copies, their scratch."""
    return 24 * 2 * ne + 200 * n + (64 << 20)


def _state_bytes(case):
    n = _size(case)[0]
    return {"construct": 0, "bfs": 64 * n, "sssp": 120 * n, "bfs_batch": (240 + 8 * case.get("roots", 0)) * n,
            "sssp_batch": 1000 * n}[case["kind"]] + (64 << 20)


def _root(dev, g, seed):
    """The first generated root with at least 4 neighbours (one in a component of a few vertices would time nothing)."""
    roots = dev.roots(g, *_seeds(seed), max_roots=16)
    rs = dev.view(g.rowstarts, (g.nlocalverts + 1,), torch.int64)
    at = torch.from_numpy(roots.astype("int64")).to(rs.device)
    degrees = (rs[at + 1] - rs[at]).cpu().numpy()
    ok = [int(r) for r, d in zip(roots, degrees) if d >= 4]
    return ok[0] if ok else int(roots[0])


def prepare(case, seed):
    n, ne = _size(case)
    kind = case["kind"]
    if kind == "generate":
        return Generate(Device(20 * ne + (1 << 20)), case, seed)
    if kind == "construct":
        return Construct(Device(20 * ne + _graph_bytes(n, ne) + (1 << 20)), case, seed)
    dev = Device(_graph_bytes(n, ne) + _state_bytes(case))
    edges = Device(20 * ne + (1 << 20))  # the tuples go when the graph is built
    g = dev.csr(_tuples(edges, case, seed), n)
    del edges
    return {"bfs": Bfs, "sssp": Sssp, "bfs_batch": BfsBatch, "sssp_batch": SsspBatch}[kind](dev, g, case, seed)


def run(state):
    return state.run()


class Generate:
    def __init__(self, dev, case, seed):
        self.dev, self.case, self.seeds = dev, case, _seeds(seed)

    def run(self):
        dev, c = self.dev, self.case
        dev.release(0)
        tg = dev.generate(c["scale"], c["edgefactor"], *self.seeds, start=c["start"], end=c["end"])
        return {"edges": dev.view(tg.edges, (tg.edges_size, 2), torch.int64),
                "weights": dev.view(tg.weights, (tg.edges_size,), torch.float32)}


class Construct:
    """Self-loops are redirected first, so that the graphs of all seeds have the same number of entries."""

    def __init__(self, dev, case, seed):
        self.dev, self.n = dev, _size(case)[0]
        self.tuples = _tuples(dev, case, seed)
        edges = dev.view(self.tuples.edges, (self.tuples.edges_size, 2), torch.int64)
        edges[:, 1] = _no_loop(edges[:, 0], edges[:, 1], self.n)
        torch.cuda.synchronize()
        self.mark = dev.mark()

    def run(self):
        dev = self.dev
        dev.release(self.mark)
        g = dev.csr(self.tuples, self.n)
        return {"rowstarts": dev.view(g.rowstarts, (self.n + 1,), torch.int64),
                "column": dev.view(g.column, (g.nlocaledges,), torch.int32),
                "weights": dev.view(g.weights, (g.nlocaledges,), torch.float32)}


class Bfs:
    def __init__(self, dev, g, case, seed):
        self.dev, self.g, self.n, self.validate = dev, g, g.nlocalverts, case["validate"]
        self.state = dev.bfs_create(g)
        self.root = _root(dev, g, seed)

    def run(self):
        dev, g, b = self.dev, self.g, self.state
        dev.bfs(g, b, self.root)
        if self.validate:
            _, errors = dev.bfs_validate(g, b, self.root)
            return {"depth": dev.view(b.dist, (self.n,), torch.int64), "errors": errors}
        depth = dev.lib.bfs_compute_dist_from_pred(C.byref(dev.ws), C.byref(g), C.byref(b), self.root)
        dev.check()
        return {"depth": dev.view(depth, (self.n,), torch.int64)}


class Sssp:
    def __init__(self, dev, g, case, seed):
        self.dev, self.g, self.n = dev, g, g.nlocalverts
        self.state = dev.sssp_create(g, case["delta"])
        self.root = _root(dev, g, seed)

    def run(self):
        self.dev.sssp(self.g, self.state, self.root)
        return {"distance": self.dev.view(self.state.dist, (self.n,), torch.float32)}


class BfsBatch:
    def __init__(self, dev, g, case, seed):
        self.dev, self.g, self.n = dev, g, g.nlocalverts
        self.roots = dev.roots(g, *_seeds(seed), max_roots=case["roots"])
        self.state = dev.batch_create(g)
        count = g500.u64()
        self.depth = dev.lib._worker_arena_push_array(C.byref(dev.ws), self.n * len(self.roots), 8, 8, C.byref(count))

    def run(self):
        dev, g, b, n = self.dev, self.g, self.state, self.n
        dev.batch(g, b, self.roots)
        for r in range(len(self.roots)):
            dev.lib.oned_graph_bfs_batch_depth(C.byref(dev.ws), C.byref(g), C.byref(b), r, self.depth + 8 * n * r)
        dev.check()
        return {"depth": dev.view(self.depth, (len(self.roots), n), torch.int64)}


class SsspBatch:
    def __init__(self, dev, g, case, seed):
        self.dev, self.g, self.n = dev, g, g.nlocalverts
        self.roots = dev.roots(g, *_seeds(seed), max_roots=case["roots"])
        # a program keeps every root's hub distance with the graph, as the server does
        self.offsets = dev.sssp_hub_distances(g, self.roots) if case["offsets"] else None
        self.state = dev.sssp_batch_create(g, case["delta"])

    def run(self):
        dev, s = self.dev, self.state
        dev.sssp_batch(self.g, s, self.roots, self.offsets)
        return {"distance": dev.view(s.dist, (len(self.roots), self.n), torch.float32)}


# ------------------------------------------------- the same answers, plainly
# The multiple recursive generator and the Kronecker edges of Graph500, and
# textbook relaxations in 64 bits, in torch.
P = (1 << 31) - 1
MASK = (1 << 64) - 1
STEP = [[107374182, 0, 0, 0, 104480], [1, 0, 0, 0, 0], [0, 1, 0, 0, 0], [0, 0, 1, 0, 0], [0, 0, 0, 1, 0]]
CHUNK = 1 << 25


def _mul(x, y):
    return [[sum(x[i][k] * y[k][j] for k in range(5)) % P for j in range(5)] for i in range(5)]


def _power(e):
    r, b = [[int(i == j) for j in range(5)] for i in range(5)], STEP
    while e:
        if e & 1:
            r = _mul(r, b)
        b, e = _mul(b, b), e >> 1
    return r


def _apply(m, s):
    return [sum(m[i][j] * s[j] for j in range(5)) % P for i in range(5)]


def _apply_all(m, s):
    out = []
    for i in range(5):
        t = torch.zeros_like(s[0])
        for j in range(5):
            if m[i][j]:
                t += s[j] * m[i][j] % P
        out.append(t % P)
    return out


def _next(s):
    z = (s[0] * 107374182 % P + s[4] * 104480 % P) % P
    return [z] + s[:4]


def _seed_state(s1, s2):
    low = (1 << 30) - 1
    return [(s1 & low) + 1, ((s1 >> 30) & low) + 1, (s2 & low) + 1, ((s2 >> 30) & low) + 1,
            ((s2 >> 60) << 4) + (s1 >> 60) + 1]


def _signed(x):
    x &= MASK
    return x - (1 << 64) if x >> 63 else x


def _reverse_bits(x):
    for shift, mask in ((1, 0x5555555555555555), (2, 0x3333333333333333), (4, 0x0F0F0F0F0F0F0F0F),
                        (8, 0x00FF00FF00FF00FF), (16, 0x0000FFFF0000FFFF), (32, 0x00000000FFFFFFFF)):
        x = ((x >> shift) & mask) | ((x & mask) << shift)
    return x


def _kronecker(scale, s1, s2, start, end):
    """Chunks (source, target, weight numerator) of the edges [start, end)."""
    seed = _seed_state(s1, s2)
    s = _apply(_power(50 * (1 << 128) + 7 * (1 << 64)), seed)
    vals = []
    for _ in range(4):
        s = _apply(STEP, s)
        vals.append(s[0])
    val0 = (vals[0] * 0xFFFFFFFF + vals[1]) & MASK
    val1 = (vals[2] * 0xFFFFFFFF + vals[3]) & MASK
    sum01, mul0, mul1 = (_signed(v) for v in (val0 + val1, val0 | 0x4519840211493211, val1 | 0x3050852102C843A5))

    def scramble(v):
        v = (v + sum01) * mul0
        v = (_reverse_bits(v) >> (64 - scale)) & ((1 << scale) - 1)
        return (_reverse_bits(v * mul1) >> (64 - scale)) & ((1 << scale) - 1)

    jump = [_power(1 << 64)]  # one edge, then doubled
    while 1 << (len(jump) - 1) < CHUNK:
        jump.append(_mul(jump[-1], jump[-1]))
    for at in range(start, end, CHUNK):
        count = min(CHUNK, end - at)
        s = [torch.tensor([z], device="cuda") for z in _apply(_power(at << 64), seed)]
        k = 0
        while len(s[0]) < count:
            s = [torch.cat(p) for p in zip(s, _apply_all(jump[k], s))]
            k += 1
        s = [z[:count].clone() for z in s]
        src, tgt = torch.zeros_like(s[0]), torch.zeros_like(s[0])
        for level in range(scale - 1, -1, -1):
            s = _next(s)
            again = (s[0] < 3647).nonzero().squeeze(1)
            while len(again):
                part = _next([z[again] for z in s])
                for z, q in zip(s, part):
                    z[again] = q
                again = again[part[0] < 3647]
            u = s[0] % 10000
            so = ((u >= 1900) & (u < 3800)) | (u >= 9500)
            to = (u < 1900) | (u >= 9500)
            swap = (src == tgt) & so & ~to
            so, to = so & ~swap, to | swap
            src += so.long() << level
            tgt += to.long() << level
        yield scramble(src), scramble(tgt), _next(s)[0]


def _edges(case, seed):
    """Chunks (source, target, weight) of a case's whole edge list."""
    if case["graph"] == "uniform":
        e, w = _uniform(case, seed)
        return [(e[:, 0].int(), e[:, 1].int(), w)]
    return [(a.int(), b.int(), z.float() * 2.0 ** -31)
            for a, b, z in _kronecker(case["scale"], *_seeds(seed), 0, _size(case)[1])]


def _shortest(n, chunks, root):
    """Distances in 64 bits by rounds of relaxations (-1: unreached)."""
    dist = torch.full((n,), math.inf, dtype=torch.float64, device="cuda")
    dist[root] = 0
    active = torch.zeros(n, dtype=torch.bool, device="cuda")
    active[root] = True
    while bool(active.any()):
        new = dist.clone()
        bits = new.view(torch.int64)  # non-negative floats order as their bits
        for a, b, w in chunks:
            for x, y in ((a, b), (b, a)):
                at = active.index_select(0, x).nonzero().squeeze(1)
                y_at = y[at].long()
                cand = dist[x[at].long()] + w[at].double()
                less = cand < new[y_at]
                bits.scatter_reduce_(0, y_at[less], cand[less].view(torch.int64), "amin")
        active, dist = new < dist, new
    return torch.where(torch.isinf(dist), -1.0, dist)


def _depths(n, chunks, root):
    depth = torch.full((n,), -1, dtype=torch.int64, device="cuda")
    depth[root] = 0
    level = 0
    while True:
        found = torch.zeros(n, dtype=torch.bool, device="cuda")
        front = depth == level
        for a, b, _ in chunks:
            for x, y in ((a, b), (b, a)):
                found[y[front.index_select(0, x)].long()] = True
        found &= depth < 0
        if not bool(found.any()):
            return depth
        level += 1
        depth[found] = level


def exact(case, seed):
    n, ne = _size(case)
    kind = case["kind"]
    if kind == "generate":
        parts = list(_kronecker(case["scale"], *_seeds(seed), case["start"], case["end"]))
        return {"edges": torch.cat([torch.stack(p[:2], 1) for p in parts]),
                "weights": torch.cat([p[2].double() for p in parts]) * 2.0 ** -31}
    if kind in ("bfs", "bfs_batch") and ne * case.get("roots", 1) > 1 << 30:
        return None  # too long: one pass over the edges per level and root
    chunks = _edges(case, seed)
    if kind == "construct":
        a, b, w = (torch.cat(p) for p in zip(*chunks))
        b = _no_loop(a, b, n)
        row, col, w = torch.cat([a, b]), torch.cat([b, a]), torch.cat([w, w])
        order = torch.sort(col, stable=True).indices
        key = (row[order].long() << 31) | w[order].view(torch.int32).long()
        order = order[torch.sort(key, stable=True).indices]
        starts = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
        starts[1:] = torch.cumsum(torch.bincount(row, minlength=n), 0)
        return {"rowstarts": starts, "column": col[order], "weights": w[order].double()}
    # roots are an input: the library's rule picks them from the graph
    state = prepare(case, seed)
    if kind == "bfs":
        out = {"depth": _depths(n, chunks, state.root)}
        return {**out, "errors": 0} if case["validate"] else out
    if kind == "sssp":
        return {"distance": _shortest(n, chunks, state.root)}
    roots = [int(r) for r in state.roots]
    del state
    if kind == "bfs_batch":
        return {"depth": torch.stack([_depths(n, chunks, r) for r in roots])}
    return {"distance": torch.stack([_shortest(n, chunks, r) for r in roots])}
