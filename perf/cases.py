"""Workloads of the dynamic-graph framework: what a program that uses it has it do.

Every case runs through the public classes of hornet_amd.graph on a seeded
graph: R-MAT (edge factor 16 unless given, symmetrized, deduplicated; the
configurations of bench.py and the tests), Chung-Lu (power-law with an odd
vertex count), or a road-like lattice (long paths, degree at most 4, the kind
of graph the DIMACS9 reader loads).  All outputs are whole numbers.

kinds:
  bfs     one BfsTopDown traversal: the distance row
  multi   one BfsMulti launch of k sources, optionally cut at a depth: k rows
  update  one step of an edge stream: insert the new batch, erase the one
          before it, read the graph back (CSR, or COO with the edge field)
  tc      one TriangleCounting2 pass: the total and the per-vertex counts
  build   a graph from its edge list (device COO, or the host CSR that a file
          reader hands over), read back as CSR
  serve   a Server replay of a burst of BFS / 2-hop queries with update
          batches between them: every request's answer
"""
import numpy as np
import torch

from hornet_amd import graph as G


def listed():
    return [
        # the smallest traversal of the tests: launches and latency
        {"name": "bfs_rmat12", "kind": "bfs", "graph": "rmat", "scale": 12, "ef": 16},
        # an ordinary graph, about a million vertices
        {"name": "bfs_rmat20", "kind": "bfs", "graph": "rmat", "scale": 20, "ef": 16},
        # the headline benchmark's graph
        {"name": "bfs_rmat24", "kind": "bfs", "graph": "rmat", "scale": 24, "ef": 16},
        # a road network: over a thousand levels, each with few vertices
        {"name": "bfs_road_733x1021", "kind": "bfs", "graph": "road", "rows": 733, "cols": 1021},
        # batched 2-hop neighbourhoods, a ragged number of sources
        {"name": "multi_cl100k_k17_2hop", "kind": "multi", "graph": "cl", "n": 99991, "avg": 16, "k": 17, "depth": 2},
        # a full batch of whole traversals
        {"name": "multi_rmat22_k64", "kind": "multi", "graph": "rmat", "scale": 22, "ef": 16, "k": 64, "depth": 0},
        # an edge stream in small batches
        {"name": "update_rmat16_1k", "kind": "update", "graph": "rmat", "scale": 16, "ef": 16, "pairs": 1000,
         "dedup": True, "sym": True, "meta": False},
        # ... in ordinary ones, a directed multigraph with a weight per edge
        {"name": "update_cl1m_100k_weights", "kind": "update", "graph": "cl", "n": 1000003, "avg": 24,
         "pairs": 100003, "dedup": False, "sym": False, "meta": True},
        # ... and the benchmark's update rounds: a million pairs each way
        {"name": "update_rmat24_1m", "kind": "update", "graph": "rmat", "scale": 24, "ef": 16, "pairs": 1 << 20,
         "dedup": True, "sym": True, "meta": False},
        # a triangle count of the four-million-vertex configuration
        {"name": "tc_rmat22", "kind": "tc", "graph": "rmat", "scale": 22, "ef": 16, "oriented": False},
        # a graph from an edge list on the device
        {"name": "build_rmat21_coo", "kind": "build", "graph": "rmat", "scale": 21, "ef": 16, "host": False},
        # a served burst: the benchmark's mix on a graph of a million vertices
        {"name": "serve_rmat20_300", "kind": "serve", "graph": "rmat", "scale": 20, "ef": 16, "requests": 300},
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi], odd more often than not."""
    x = int(round(lo * (hi / lo) ** rng.random()))
    return min(max(x | 1 if rng.random() < 0.7 else x, lo), hi)


def _draw_graph(rng, max_scale, road):
    kind = rng.choice(["rmat", "rmat", "cl"] + (["road"] if road else []))
    if kind == "rmat":
        scale = rng.randint(10, max_scale)
        return {"graph": "rmat", "scale": scale, "ef": 16 if scale == max_scale else rng.choice([7, 11, 16])}
    if kind == "cl":
        return {"graph": "cl", "n": _log(rng, 1000, 1 << max(max_scale - 1, 11)), "avg": rng.choice([9, 16, 24])}
    return {"graph": "road", "rows": _log(rng, 20, 733), "cols": _log(rng, 20, 1021)}


def draw(rng):
    kind = rng.choice(["bfs", "bfs", "multi", "update", "update", "tc", "build", "serve"])
    c = {"kind": kind}
    if kind == "bfs":
        c.update(_draw_graph(rng, 24, True))
    elif kind == "multi":
        c.update(_draw_graph(rng, 21, False))
        c.update(k=rng.randint(1, 64), depth=rng.choice([0, 0, 2, 3]))
    elif kind == "update":
        c.update(_draw_graph(rng, 23, True))
        sym = rng.random() < 0.6
        top = {"rmat": 1 << c.get("scale", 0), "cl": c.get("n", 0), "road": c.get("rows", 0) * c.get("cols", 0)}
        c.update(pairs=_log(rng, 100, max(min(1 << 20, top[c["graph"]]), 200)), dedup=sym or rng.random() < 0.5,
                 sym=sym, meta=rng.random() < 0.3)
    elif kind == "tc":
        c.update(_draw_graph(rng, 21, False))   # a lattice has no triangles
        c.update(oriented=rng.random() < 0.3)
    elif kind == "build":
        c.update(_draw_graph(rng, 21, True))
        c.update(host=c.get("scale", 0) <= 18 and rng.random() < 0.4)
    else:
        c.update({"graph": "rmat", "scale": rng.randint(12, 19), "ef": 16, "requests": _log(rng, 20, 300)})
    return c


# ------------------------------------------------------------------ inputs
def _nv(c):
    if c["graph"] == "rmat":
        return 1 << c["scale"]
    return c["n"] if c["graph"] == "cl" else c["rows"] * c["cols"]


def _lattice(c):
    """Every street of the lattice once."""
    v = torch.arange(c["rows"] * c["cols"], dtype=torch.int32, device="cuda").view(c["rows"], c["cols"])
    return torch.cat([v[:, :-1].reshape(-1), v[:-1].reshape(-1)]), torch.cat([v[:, 1:].reshape(-1), v[1:].reshape(-1)])


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _pairs(c, seed, count=None):
    """The graph's edge list on the device, each undirected edge once (repeats and loops included)."""
    if c["graph"] == "rmat":
        return G.rmat_pairs_device(c["scale"], seed, c["ef"], 0, count)
    if c["graph"] == "cl":
        return G.chung_lu_pairs_device(c["n"], count or c["n"] * c["avg"] // 2, seed)
    src, dst = _lattice(c)
    keep = torch.rand(src.numel(), generator=_gen(seed), device="cuda") < 0.9   # one street in ten is closed
    return src[keep].contiguous(), dst[keep].contiguous()


def _graph(c, seed):
    return G.Hornet.from_coo_device(_nv(c), *_pairs(c, seed))


def _sources(h, k, seed):
    """k seeded vertices with at least one edge."""
    nz = torch.nonzero(h.degrees()).view(-1).cpu().numpy()
    return nz[np.random.default_rng(seed).integers(0, nz.size, k)].astype(np.int32)


def _edge_count(c):
    """Undirected edges of the graphs whose size does not depend on the seed."""
    if c["graph"] == "road":
        full = c["rows"] * (c["cols"] - 1) + (c["rows"] - 1) * c["cols"]
        return int(0.9 * full)
    if c["graph"] == "rmat":
        return int(0.95 * c["ef"] * _nv(c))
    return int(0.9 * c["avg"] * c["n"] / 2)


def _keys(c, src, dst):
    """Canonical keys (smaller end * nv + larger end) of the pairs that are no loops, sorted, each once."""
    keep = src != dst
    src, dst = src[keep].long(), dst[keep].long()
    return torch.unique(torch.minimum(src, dst) * _nv(c) + torch.maximum(src, dst))


def _edges(c, seed):
    """Exactly _edge_count(c) undirected edges as sorted keys: a larger sample, thinned."""
    want = _edge_count(c)
    if c["graph"] == "road":
        k = _keys(c, *_lattice(c))
    else:
        count = int(1.15 * want) + 64
        k = _keys(c, *_pairs(c, seed, count))
        while k.numel() < want:
            count *= 2
            k = _keys(c, *_pairs(c, seed, count))
    return _thin(k, want, seed)


def _thin(k, want, seed):
    """`want` of the sorted keys, the others left out at even distances from a seeded start."""
    n, drop = k.numel(), k.numel() - want
    if drop <= 0:
        return k
    at = (torch.arange(drop, device="cuda", dtype=torch.float64) + torch.rand(1, generator=_gen(seed), device="cuda").double()) * (n / drop)
    keep = torch.ones(n, dtype=torch.bool, device="cuda")
    keep[at.long().clamp_(max=n - 1)] = False
    return k[keep][:want]


def _both(c, k):
    """Keys to pairs of either direction."""
    u, v = (k // _nv(c)).int(), (k % _nv(c)).int()
    return torch.cat([u, v]), torch.cat([v, u])


def _batches(c, edges, seed):
    """Two batches of an edge stream: uniform pairs that the graph does not hold, in random order and direction,
    with one repeat in a hundred; both directions of each when symmetric, with a weight per entry if there is a field."""
    n, nv = c["pairs"], _nv(c)
    have, count = 0, int(2.2 * n) + 64
    while have < 2 * n:
        k = _keys(c, *G.uniform_pairs_device(nv, count, seed))
        at = torch.searchsorted(edges, k).clamp_(max=edges.numel() - 1)
        k = k[edges[at] != k]
        have, count = k.numel(), 2 * count
    k = k[torch.randperm(have, generator=_gen(seed), device="cuda")[: 2 * n]]
    out = []
    for part in (k[:n], k[n:]):
        again = torch.randint(0, n, (n // 100,), generator=_gen(seed + 1), device="cuda")
        u, v = (part // nv).int(), (part % nv).int()
        turn = torch.rand(n, generator=_gen(seed + 2), device="cuda") < 0.5
        s, d = torch.where(turn, v, u), torch.where(turn, u, v)
        s, d = torch.cat([s, s[again]]), torch.cat([d, d[again]])
        if c["sym"]:
            s, d = torch.cat([s, d]), torch.cat([d, s])
        w = [np.random.default_rng(seed).integers(1, 1000, s.numel()).astype(np.int32)] if c["meta"] else None
        out.append(G.BatchUpdate(s, d, meta=w))
    return out


def _trace(h, c, seed):
    """A burst: 70 % BFS, 20 % 2-hop, 10 % updates of 100 to 30,000 pairs; every batch inserted is erased later on."""
    rng, order = np.random.default_rng(seed), np.random.default_rng(c["requests"])
    nz = torch.nonzero(h.degrees()).view(-1).cpu().numpy()
    trace, live = [], []
    for k in order.choice(3, c["requests"], p=[0.7, 0.2, 0.1]):
        if k < 2:
            trace.append((G.Server.BFS if k == 0 else G.Server.TWO_HOP, int(nz[rng.integers(0, nz.size)])))
        elif live and order.random() < 0.5:
            trace.append((G.Server.ERASE, live.pop(0)))
        else:
            s, d = rng.integers(0, h.nV(), (2, int(10 ** order.uniform(2, 4.5)))).astype(np.int32)
            s, d = s[s != d], d[s != d]
            live.append((np.concatenate([s, d]), np.concatenate([d, s])))
            trace.append((G.Server.INSERT, live[-1]))
    return trace + [(G.Server.ERASE, b) for b in live]


def _file_csr(c, seed):
    """A host CSR as a file reader hands it over: rows in file order, not sorted."""
    src, dst = _both(c, _edges(c, seed))
    order = torch.randperm(src.numel(), generator=_gen(seed), device="cuda")
    src, dst = src[order], dst[order]
    at = torch.argsort(src, stable=True)
    off = torch.zeros(_nv(c) + 1, dtype=torch.int64, device="cuda")
    off[1:] = torch.bincount(src.long(), minlength=_nv(c)).cumsum(0)
    return off.cpu().numpy(), dst[at].cpu().numpy()


def _edge_list(c, seed):
    """A device edge list as collected: random order and directions, one edge in twelve repeated, some loops."""
    k = _edges(c, seed)
    g = _gen(seed)
    again = torch.randint(0, k.numel(), (k.numel() // 12,), generator=g, device="cuda")
    loop = torch.randint(0, _nv(c), (k.numel() // 100,), generator=g, device="cuda") * (_nv(c) + 1)
    k = torch.cat([k, k[again], loop])
    k = k[torch.randperm(k.numel(), generator=g, device="cuda")]
    u, v = (k // _nv(c)).int(), (k % _nv(c)).int()
    turn = torch.rand(k.numel(), generator=g, device="cuda") < 0.5
    return torch.where(turn, v, u), torch.where(turn, u, v)


def prepare(case, seed):
    c = case
    if c["kind"] == "build":
        if c["host"]:
            off, adj = _file_csr(c, seed)
            return {"c": c, "off": off, "adj": adj}
        src, dst = _edge_list(c, seed)
        return {"c": c, "src": src, "dst": dst}
    if c["kind"] == "update":
        edges = _edges(c, seed)
        h = G.Hornet.from_coo_device(_nv(c), *((edges // _nv(c)).int(), (edges % _nv(c)).int()))
        old, new = _batches(c, edges, seed)
        del edges
        if c["meta"]:
            off, adj = h.getCSR()
            w = torch.randint(1, 1000, (adj.numel(),), generator=_gen(seed), device="cuda", dtype=torch.int32)
            h = G.Hornet.from_device_csr(off, adj, meta=[w])
        h.insert(old, c["dedup"], c["dedup"])
        return {"c": c, "h": h, "batches": [old, new]}
    h = _graph(c, seed)
    if c["kind"] == "bfs":
        bfs = G.BfsTopDown(h)
        bfs.set_parameters(int(_sources(h, 1, seed)[0]))
        return {"c": c, "bfs": bfs}
    if c["kind"] == "multi":
        limits = np.full(c["k"], c["depth"], np.int32) if c["depth"] else None
        return {"c": c, "multi": G.BfsMulti(h), "sources": _sources(h, c["k"], seed), "limits": limits}
    if c["kind"] == "tc":
        if c["oriented"]:
            s, d = h.getCOO()
            deg = h.degrees()
            ds, dd = deg[s.long()], deg[d.long()]
            keep = (ds < dd) | ((ds == dd) & (s < d))
            off = torch.zeros(h.nV() + 1, dtype=torch.int64, device="cuda")
            off[1:] = torch.bincount(s[keep].long(), minlength=h.nV()).cumsum(0)
            h = G.Hornet.from_device_csr(off, d[keep])
        tc = G.TriangleCounting2(h)
        tc.init()
        return {"c": c, "tc": tc}
    return {"c": c, "h": h, "server": G.Server(h), "trace": _trace(h, c, seed)}


# ------------------------------------------------------------------ one pass
def run(state):
    kind = state["c"]["kind"]
    if kind == "bfs":
        state["bfs"].run()
        return state["bfs"].distances()
    if kind == "multi":
        return state["multi"].run(state["sources"], state["limits"])
    if kind == "update":
        h, (old, new), dedup = state["h"], state["batches"], state["c"]["dedup"]
        added = h.insert(new, dedup, dedup)
        removed = h.erase(old, dedup)
        state["batches"] = [new, old]   # the stream's next step
        return added, removed, h.getCOO(meta=True) if state["c"]["meta"] else h.getCSR()
    if kind == "tc":
        tc = state["tc"]
        if state["c"]["oriented"]:
            tc.run()
        else:
            tc.run_undirected()
        return tc.countTriangles(), tc.triPerVertex
    if kind == "build":
        if state["c"]["host"]:
            h = G.Hornet.from_csr(state["off"], state["adj"])
        else:
            h = G.Hornet.from_coo_device(_nv(state["c"]), state["src"], state["dst"])
        return h.getCSR()
    n = len(state["trace"])
    res = state["server"].replay(state["trace"], np.zeros(n, np.int64))[-n:]
    return {f: res[f] for f in ("status", "reached", "dist_sum", "max_depth", "applied")}


def work(case):
    """Bytes that one pass cannot do without: each entry and record it needs read once, each result written once."""
    c = case
    nv = _nv(c)
    m = 2 * _edge_count(c)               # stored (directed) entries
    if c["kind"] == "bfs":
        return {"bytes": 4 * m + 16 * nv + 4 * nv, "flops": 0}
    if c["kind"] == "multi":
        return {"bytes": 4 * m + 16 * nv + 4 * nv * c["k"], "flops": 0}
    if c["kind"] == "update":
        b = c["pairs"] * (2 if c["sym"] else 1)
        touched = min(b, nv)
        field = 4 if c["meta"] else 0
        # both batches read, their vertices' records and rows read and written, the graph read back
        return {"bytes": 2 * (8 * b + (32 + 2 * (4 + field) * m / nv) * touched) + 16 * nv + 2 * (4 + field) * m,
                "flops": 0}
    if c["kind"] == "tc":
        return {"bytes": 4 * m + 16 * nv + 8 * nv, "flops": 0}
    if c["kind"] == "build":
        return {"bytes": (4 * m + 8 * nv if c["host"] else 4.4 * m) + 4 * m + 16 * nv + 4 * m + 8 * nv, "flops": 0}
    # one traversal's reads for every 64 queries, and the update batches
    return {"bytes": (c["requests"] / 64 + 1) * (4 * m + 16 * nv) + 0.1 * c["requests"] * 6000 * 16, "flops": 0}
