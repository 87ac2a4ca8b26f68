"""GPU parity of the BFS level steps at the sizes where each can go wrong:
graphs traversed by one launch, levels run by one workgroup (bitmap in LDS and
in memory, frontiers that outgrow LDS), whole-device pushes, and bottom-up
levels with rows settled by a lane, by a team and by the whole workgroup."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
INF = 2**31 - 1


@pytest.fixture(scope="module")
def hn():
    import hornet_amd.graph as G
    return G


def device_graph(hn, n, s, d):
    """The symmetric simple graph of the pairs, known to be symmetric, and its host CSR."""
    import torch
    s, d = np.asarray(s, np.int32), np.asarray(d, np.int32)
    h = hn.Hornet.from_coo_device(n, torch.from_numpy(s).cuda(), torch.from_numpy(d).cuda())
    off, adj = h.getCSR()
    return h, off.cpu().numpy(), adj.cpu().numpy()


def check(hn, h, off, adj, sources):
    bfs = hn.BfsTopDown(h)
    for src in sources:
        print(f"  source {src}", flush=True)
        exp, scanned = O.bfs(off, adj, int(src))
        bfs.set_parameters(int(src))
        for _ in range(2):   # the second one queues as many rounds as the first needed
            bfs.run()
            assert np.array_equal(bfs.distances().cpu().numpy(), exp), src
            assert bfs.stats.visited == int((exp != INF).sum())
            assert bfs.stats.edges_scanned == scanned
            assert bfs.stats.levels == int(exp[exp != INF].max()) + 1


def lattice(rows, cols, seed):
    v = np.arange(rows * cols).reshape(rows, cols)
    s = np.concatenate([v[:, :-1].ravel(), v[:-1].ravel()])
    d = np.concatenate([v[:, 1:].ravel(), v[1:].ravel()])
    keep = np.random.default_rng(seed).random(s.size) < 0.9
    return s[keep], d[keep]


# 8192 vertices and 2^18 entries bound the graphs that one launch traverses
@pytest.mark.parametrize("n,m", [(2, 1), (33, 40), (8191, 60000), (8192, 60000), (8192, 131300), (8193, 60000)])
def test_uniform_around_the_one_launch_limit(hn, n, m):
    print(f"case bfs uniform n={n} m={m}", flush=True)
    s, d = np.random.default_rng(n + m).integers(0, n, (2, m))
    h, off, adj = device_graph(hn, n, s, d)
    check(hn, h, off, adj, O.pick_sources(off, 3, seed=1) if adj.size else [0])


# the last three: frontiers above 4096 vertices, and bitmaps just in and out of LDS (770,048 vertices)
@pytest.mark.parametrize("rows,cols", [(2, 5000), (97, 101), (3000, 256), (3008, 256), (3009, 256)])
def test_lattices(hn, rows, cols):
    print(f"case bfs lattice {rows}x{cols}", flush=True)
    h, off, adj = device_graph(hn, rows * cols, *lattice(rows, cols, 5))
    check(hn, h, off, adj, [int(rows // 2 * cols + cols // 2)] + O.pick_sources(off, 1, seed=2).tolist())


def test_frontier_outgrows_one_workgroup(hn):
    # a hub of 70,000 leaves, each with a leaf of its own: the frontier jumps
    # from one vertex past the LDS list and back to nothing
    print("case bfs broom", flush=True)
    k = 70000
    s = np.concatenate([np.zeros(k), np.arange(1, k + 1), [2 * k + 1, 2 * k + 2]])
    d = np.concatenate([np.arange(1, k + 1), np.arange(k + 1, 2 * k + 1), [2 * k + 2, 0]])
    h, off, adj = device_graph(hn, 2 * k + 5, s, d)
    check(hn, h, off, adj, [0, 2 * k + 1, k + 7, 2 * k + 4])


# (the last takes the longer spans)
@pytest.mark.parametrize("n,deg", [(20011, 64), (700001, 16), (3300007, 8)])
def test_bottom_up_levels(hn, n, deg):
    """Uniform random graphs reach most vertices in one level (a pull); every
    fifth vertex has no edges, and a separate component stays unreached."""
    print(f"case bfs bottom-up n={n}", flush=True)
    rng = np.random.default_rng(n)
    live = np.flatnonzero(np.arange(n) % 5 != 2)
    core, rest = live[: live.size * 9 // 10], live[live.size * 9 // 10:]
    s = np.concatenate([core[rng.integers(0, core.size, n * deg // 2)], rest[:-1]])
    d = np.concatenate([core[rng.integers(0, core.size, n * deg // 2)], rest[1:]])
    h, off, adj = device_graph(hn, n, s, d)
    check(hn, h, off, adj, [int(core[0]), int(core[-1]), int(rest[0])] if n < 10**6 else [int(core[5])])


@pytest.mark.parametrize("leaves", [3, 4, 5, 11, 12, 13, 29, 33, 511, 513, 2049, 16895, 16897, 40000])
def test_bottom_up_long_rows(hn, leaves):
    """Hubs whose one reached neighbour comes last in their row, after leaves
    that are reached through the hub only: settled by a lane, a team, or the
    whole workgroup; one hub more is not connected at all."""
    print(f"case bfs long rows leaves={leaves}", flush=True)
    rng = np.random.default_rng(leaves)
    hubs = 70 if leaves < 5000 else 12
    n0 = hubs * leaves
    ncore = 30000
    core = n0 + rng.integers(0, ncore, (2, ncore * 24))
    hub = n0 + ncore + np.arange(hubs)
    s = np.concatenate([core[0], np.repeat(hub, leaves), hub[:-1]])
    d = np.concatenate([core[1], np.arange(n0), n0 + rng.integers(0, ncore, hubs - 1)])
    h, off, adj = device_graph(hn, n0 + ncore + hubs + 3, s, d)
    check(hn, h, off, adj, [n0 + 1, n0 + 77, 0, int(hub[-1])])


def test_directed_graphs_never_pull(hn):
    print("case bfs directed", flush=True)
    import torch
    n = 30000
    s, d = np.random.default_rng(3).integers(0, n, (2, n * 24)).astype(np.int32)
    keep = s < d
    h = hn.Hornet.from_coo_device(n, torch.from_numpy(s[keep]).cuda(), torch.from_numpy(d[keep]).cuda(),
                                  symmetrize=False)
    off, adj = (x.cpu().numpy() for x in h.getCSR())
    check(hn, h, off, adj, [0, 5, n // 2])
