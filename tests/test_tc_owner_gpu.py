"""GPU parity of triangle counting where the owner's LDS set, its hash passes,
its tasks and the short lists meet their limits."""
from math import comb

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hn():
    import hornet_amd.graph as G
    return G


def run(hn, h, stored):
    tc = hn.TriangleCounting2(h)
    tc.init()
    for _ in range(2):   # the second one on dirty scratch
        (tc.run if stored else tc.run_undirected)()
    return tc.countTriangles(), tc.copyTCToHost()


def complete(n):
    s, d = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
    m = s != d
    return O.coo_to_csr(n, s[m].astype(np.int32), d[m].astype(np.int32))


# oriented lists reach n - 1 entries: short lists end at 16, hashed passes and teams at 512 and 256
@pytest.mark.parametrize("n", [3, 4, 5, 16, 17, 18, 19, 33, 65, 258, 514])
def test_complete_graphs(hn, n):
    print(f"case tc K{n}", flush=True)
    off, adj = complete(n)
    h = hn.Hornet.from_csr(off, adj)
    total, per = run(hn, h, False)
    do, da = O.directed_by_degree(off, adj)
    assert total == comb(n, 3) and np.array_equal(per, O.tc2_per_vertex(do, da))
    total, per = run(hn, h, True)
    assert total == 6 * comb(n, 3) and np.array_equal(per, O.tc2_per_vertex(off, adj))


def test_no_hubs_and_two_hash_passes(hn):
    """190 cliques of 700: 133,000 vertices of one degree are too many to be
    hubs, so that every list, up to 699 entries, is hashed, in two passes."""
    import torch
    print("case tc cliques", flush=True)
    n, k = 700, 190
    off, adj = complete(n)
    src = np.repeat(np.arange(n), np.diff(off))
    up = src < adj
    s, d = torch.from_numpy(src[up].astype(np.int32)).cuda(), torch.from_numpy(adj[up]).cuda()
    at = (torch.arange(k, dtype=torch.int32, device="cuda") * n).view(-1, 1)
    h = hn.Hornet.from_coo_device(n * k, (s + at).view(-1), (d + at).view(-1))
    total, per = run(hn, h, False)
    do, da = O.directed_by_degree(off, adj)
    one = O.tc2_per_vertex(do, da)
    assert total == k * comb(n, 3)
    assert np.array_equal(per.reshape(k, n), np.broadcast_to(one, (k, n)))


@pytest.mark.parametrize("scale,ef", [(11, 3), (15, 16), (18, 20)])
def test_mixed_hubs_and_tails(hn, scale, ef):
    """s18: 262,144 vertices, so that lists mix hubs and others."""
    print(f"case tc rmat s{scale} ef{ef}", flush=True)
    h = hn.Hornet.rmat(scale, 9, edge_factor=ef)
    off, adj = (x.cpu().numpy() for x in h.getCSR())
    T = O.checker_threads()
    do, da = O.directed_by_degree(off, adj)
    total, per = run(hn, h, False)
    assert total == O.triangles(off, adj, threads=T)
    assert np.array_equal(per, O.tc2_per_vertex(do, da))
    ho = hn.Hornet.from_csr(do, da)
    total2, per2 = run(hn, ho, True)
    assert total2 == total and np.array_equal(per2, per)


@pytest.mark.parametrize("seed", [1, 2])
def test_stored_directed_graph(hn, seed):
    """Any stored simple graph: directed both ways here and there, self loops, rows of one entry."""
    print(f"case tc stored directed seed={seed}", flush=True)
    rng = np.random.default_rng(seed)
    n, m = 900, 40000
    s = np.concatenate([rng.integers(0, n, m), rng.integers(0, 30, m)]).astype(np.int32)
    d = np.concatenate([rng.integers(0, n, m), rng.integers(0, n, m)]).astype(np.int32)
    lone = np.arange(n, n + 50, dtype=np.int32)
    s, d = np.concatenate([s, lone]), np.concatenate([d, lone - 40])
    off, adj = O.coo_to_csr(n + 50, s, d, symmetrize=False, drop_self_loops=False, dedup=True)
    h = hn.Hornet.from_csr(off, adj)
    total, per = run(hn, h, True)
    exp = O.tc2_per_vertex(off, adj)
    assert total == int(exp.sum()) and np.array_equal(per, exp)


def test_star_of_cliques_many_tasks(hn):
    """An owner with far more edges than a task holds: 300 of a hub's
    neighbours form a clique, 5,000 more hang off that clique's vertices."""
    print("case tc many tasks", flush=True)
    rng = np.random.default_rng(4)
    core, rest = 300, 5000
    i, j = np.triu_indices(core, 1)
    s = np.concatenate([i, np.repeat(np.arange(core, core + rest), 24)])
    d = np.concatenate([j, rng.integers(0, core, rest * 24)])
    off, adj = O.coo_to_csr(core + rest, s.astype(np.int32), d.astype(np.int32), symmetrize=True, dedup=True)
    h = hn.Hornet.from_csr(off, adj)
    total, per = run(hn, h, False)
    do, da = O.directed_by_degree(off, adj)
    assert total == O.triangles(off, adj) and np.array_equal(per, O.tc2_per_vertex(do, da))


@pytest.mark.parametrize("both", [True, False])
def test_long_lists_of_ids(hn, both):
    """Stars of 510 to 514 leaves and one of 5,000, the leaves of each in a ring
    with its second neighbours: 70,000 vertices of one frequency, too many to be
    hubs, so that rows on both sides of 512 hold ids only.  The leaves name
    their centre or not."""
    print(f"case tc long id lists both={both}", flush=True)
    sizes = [510 + i % 5 for i in range(128)] + [5000]
    src, dst, n = [], [], 0
    for k in sizes:
        leaf = n + 1 + np.arange(k)
        src.append(np.full(k, n)), dst.append(leaf)
        if both:
            src.append(leaf), dst.append(np.full(k, n))
        for d in (1, 2, k - 1, k - 2):
            src.append(leaf), dst.append(n + 1 + (np.arange(k) + d) % k)
        n += k + 1
    off, adj = O.coo_to_csr(n, np.concatenate(src).astype(np.int32), np.concatenate(dst).astype(np.int32))
    h = hn.Hornet.from_csr(off, adj)
    total, per = run(hn, h, True)
    exp = O.tc2_per_vertex(off, adj)
    assert total == int(exp.sum()) and np.array_equal(per, exp)


def test_oriented_lists_of_ids(hn):
    """66 cliques of 1,000 and one of 1,100: 67,100 vertices with too many of a
    degree to be hubs, whose oriented lists lie on both sides of 512."""
    import torch
    print("case tc oriented id lists", flush=True)
    src, dst, n = [], [], 0
    for k in [1000] * 66 + [1100]:
        i, j = np.triu_indices(k, 1)
        src.append((i + n).astype(np.int32)), dst.append((j + n).astype(np.int32))
        n += k
    h = hn.Hornet.from_coo_device(n, torch.from_numpy(np.concatenate(src)).cuda(),
                                  torch.from_numpy(np.concatenate(dst)).cuda())
    total, per = run(hn, h, False)
    exp = []
    for k in (1000, 1100):
        off, adj = complete(k)
        exp.append(O.tc2_per_vertex(*O.directed_by_degree(off, adj)))
    assert total == 66 * comb(1000, 3) + comb(1100, 3)
    assert np.array_equal(per[:66000].reshape(66, 1000), np.broadcast_to(exp[0], (66, 1000)))
    assert np.array_equal(per[66000:], exp[1])


@pytest.mark.parametrize("n", [1 << 20, (1 << 20) + 37])
def test_short_lists_of_many_vertices(hn, n):
    """Both sides of where a wave takes 64 vertices instead of 16: a strip of
    triangles with gaps, so that sources are few, many or none among a wave's."""
    print(f"case tc short lists n={n}", flush=True)
    i = np.arange(n - 2, dtype=np.int32)
    i = i[(i // 300) % 3 != 1]
    i = np.concatenate([i[: i.size // 2], i[i.size // 2 :][::7], [n - 3]]).astype(np.int32)
    s, d = np.concatenate([i, i, i + 1]), np.concatenate([i + 1, i + 2, i + 2])
    off, adj = O.coo_to_csr(n, s, d, symmetrize=True, dedup=True)
    h = hn.Hornet.from_csr(off, adj)
    total, per = run(hn, h, False)
    do, da = O.directed_by_degree(off, adj)
    exp = O.tc2_per_vertex(do, da)
    assert total == int(exp.sum()) and np.array_equal(per, exp)
    total, per = run(hn, h, True)
    exp = O.tc2_per_vertex(off, adj)
    assert total == int(exp.sum()) and np.array_equal(per, exp)
