"""Triangle counts whose owners' ids take more than one hash table: 256 ids beside
the hubs' bits, then 1,024 at a time in their place; stored rows of more than 2,304
are searched.  Ids are kept from being hubs by there being more than 65,535 vertices
of their weight."""
from math import comb

import numpy as np
import pytest

import oracle as O

gpu = pytest.mark.gpu


@pytest.fixture(scope="module")
def hn():
    import hornet_amd.graph as G
    return G


def run(hn, h, stored):
    tc = hn.TriangleCounting2(h)
    tc.init()
    got = []
    for _ in range(2):   # the second one on dirty scratch
        (tc.run if stored else tc.run_undirected)()
        got.append((tc.countTriangles(), tc.copyTCToHost()))
    assert got[0][0] == got[1][0] and np.array_equal(got[0][1], got[1][1])
    return got[1]


def tile(n, k, off, adj):
    """k copies of a graph of n vertices"""
    deg = np.tile(np.diff(off), k)
    return (np.concatenate([[0], np.cumsum(deg)]),
            (np.tile(adj, k).reshape(k, -1) + np.arange(k)[:, None] * n).ravel().astype(np.int32))


def complete(n, times=1):
    a = np.tile(np.arange(n), (n, 1))
    a = a[~np.eye(n, dtype=bool)]
    return np.arange(n + 1) * (n - 1) * times, np.repeat(a, times)


# oriented lists of ids alone, up to n - 1 of them: one table, one and one entry, two and one
@gpu
@pytest.mark.parametrize("n,k", [(1025, 64), (1026, 64), (2050, 32)])
def test_cliques(hn, n, k):
    print(f"case tc tables K{n} x {k}", flush=True)
    h = hn.Hornet.from_csr(*tile(n, k, *complete(n)))
    total, per = run(hn, h, False)
    j = np.arange(n, dtype=np.uint64)
    assert n * k > 65535 and total == k * comb(n, 3)
    assert np.array_equal(per.reshape(k, n), np.broadcast_to(j * (n - 1 - j), (k, n)))


@gpu
def test_cliques_with_hubs(hn):
    """48 cliques of 1,400 joined to 300 hubs: lists of the hubs and 0 to 1,399 ids."""
    import torch
    print("case tc tables hubs and ids", flush=True)
    n, k, m = 1400, 48, 300
    i, j = np.triu_indices(n, 1)
    at = torch.arange(k, dtype=torch.int32, device="cuda").view(-1, 1) * n
    both = [torch.from_numpy(x.astype(np.int32)).cuda() + at for x in (i, j)]
    v = torch.arange(n * k, dtype=torch.int32, device="cuda")
    hubs = n * k + torch.arange(m, dtype=torch.int32, device="cuda")
    src = torch.cat([both[0].view(-1), v.repeat_interleave(m)])
    dst = torch.cat([both[1].view(-1), hubs.repeat(n * k)])
    h = hn.Hornet.from_coo_device(n * k + m, src, dst)
    del src, dst, both
    total, per = run(hn, h, False)
    q = np.arange(n, dtype=np.uint64)
    one = q * (n - 1 - q + m)
    assert total == k * int(one.sum()) and not per[n * k:].any()
    assert np.array_equal(per[:n * k].reshape(k, n), np.broadcast_to(one, (k, n)))


def member_counts(off, adj):
    """Per edge (u, v), u != v, of a source with two entries or more: the entries of the
    shorter list that the longer one holds, however often, for the shorter one's vertex."""
    per = np.zeros(off.size - 1, np.uint64)
    rows = [adj[off[v]:off[v + 1]] for v in range(off.size - 1)]
    for u in np.flatnonzero(np.diff(off) >= 2):
        for v, often in zip(*np.unique(rows[u], return_counts=True)):
            if v != u and rows[v].size:
                s, l, c = (rows[u], rows[v], u) if rows[u].size < rows[v].size else (rows[v], rows[u], v)
                per[c] += np.uint64(often * np.isin(s, l).sum())
    return per


@gpu
@pytest.mark.parametrize("times", [1, 3])
def test_stored_rows_with_hubs(hn, times):
    """Stored rows of 30 hubs and a number of ids on both sides of each limit; two more
    rows each that share half of the ids and some hubs, linked both ways.  65,600 more
    vertices are entries as often as an id is.  times: every entry that often."""
    print(f"case tc tables stored rows times={times}", flush=True)
    rng = np.random.default_rng(5)
    counts = [3, 200, 255, 256, 257, 1023, 1279, 1280, 1281, 2303, 2304, 2305, 2400, 2600]
    hubs, n, lists = np.arange(30), 30, {}
    for c in counts:
        a, b, z = n, n + 1, n + 2
        ids = n + 3 + np.arange(c - 2)   # b and z are entries of a as well
        n = int(ids[-1]) + 1
        lists[a] = np.concatenate([hubs, ids, [b, z]])
        lists[b] = np.concatenate([hubs[::2], ids[::2], [a, z]])
        lists[z] = np.concatenate([hubs[1::3], ids[1::2], [a]])
    fill = n + np.arange(65600)
    n += 65602
    lists[n - 1] = lists[n - 2] = fill   # (they share nothing with the ones above)
    for h in hubs:
        lists[int(h)] = rng.choice(fill, 10, replace=False)
    s = np.concatenate([np.full(e.size, v) for v, e in lists.items()])
    d = np.concatenate(list(lists.values()))
    order = np.lexsort((d, s))
    s, d = np.repeat(s[order], times), np.repeat(d[order], times).astype(np.int32)
    assert d.size < 1 << 19   # (every entry counts towards the hubs)
    off = np.concatenate([[0], np.cumsum(np.bincount(s, minlength=n))])
    exp = member_counts(off, d)
    if times == 1:
        assert np.array_equal(exp, O.tc2_per_vertex(off, d))
    h = hn.Hornet.from_csr(off, d)
    total, per = run(hn, h, True)
    assert total == int(exp.sum()) and np.array_equal(per, exp)


@gpu
@pytest.mark.parametrize("stored", [True, False])
def test_cliques_with_repeats(hn, stored):
    """190 cliques of 350, every entry three times: up to 1,047 ids of 349 vertices."""
    print(f"case tc tables repeats stored={stored}", flush=True)
    n, k = 350, 190
    h = hn.Hornet.from_csr(*tile(n, k, *complete(n, 3)))
    total, per = run(hn, h, stored)
    j = np.arange(n, dtype=np.uint64)
    one = np.full(n, 9 * (n - 1) * (n - 2), np.uint64) if stored else 9 * j * (n - 1 - j)
    assert total == k * int(one.sum())
    assert np.array_equal(per.reshape(k, n), np.broadcast_to(one, (k, n)))


def test_closed_forms_of_cliques():
    """The sums above against the definition."""
    n = 12
    off, adj = complete(n, 3)
    assert np.array_equal(member_counts(off, adj), np.full(n, 9 * (n - 1) * (n - 2)))
    src = np.repeat(np.arange(n), np.diff(off))
    up = src < adj
    j = np.arange(n)
    o = np.concatenate([[0], np.cumsum(np.bincount(src[up], minlength=n))])
    assert np.array_equal(member_counts(o, adj[up]), 9 * j * (n - 1 - j))
