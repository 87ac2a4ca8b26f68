"""Batched BFS where its level codes and its first look at a row meet their limits:
levels on both sides of the last code, counts of sources on both sides of the rule,
vertex counts that fill no quad, rows as long as the first look."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
INF = 2**31 - 1


@pytest.fixture(scope="module")
def hn():
    import hornet_amd.graph as G
    return G


def expected(off, adj, srcs, limits=None):
    d = np.stack([O.bfs(off, adj, int(s))[0] for s in srcs])
    if limits is not None:
        for i, l in enumerate(limits):
            if l > 0:
                d[i][d[i] > l] = INF
    return d


@pytest.mark.parametrize("n", [13, 14, 15, 16, 17, 18, 66, 257])
@pytest.mark.parametrize("k", [1, 7, 8, 64])
def test_paths(hn, n, k):
    print("case msbfs path", n, k, flush=True)
    v = np.arange(n - 1, dtype=np.int32)
    off, adj = O.coo_to_csr(n + 2, v, v + 1)   # two vertices that no path reaches
    h = hn.Hornet.from_csr(off, adj)
    srcs = np.resize(np.array([0, n - 1, n // 2, n, 0], dtype=np.int32), k)
    ms = hn.BfsMulti(h)
    for _ in range(2):
        assert np.array_equal(ms.run(srcs).cpu().numpy(), expected(off, adj, srcs))


@pytest.mark.parametrize("deg", [1, 3, 4, 5, 7, 8, 9, 12, 33])
@pytest.mark.parametrize("alpha", [1, 1 << 20])
def test_row_lengths(hn, deg, alpha):
    print("case msbfs rows", deg, alpha, flush=True)
    n = 1001
    rng = np.random.default_rng(deg)
    s = np.repeat(np.arange(n), deg)
    d = (s + np.tile(1 + rng.permutation(n - 1)[:deg], n)) % n
    off, adj = O.coo_to_csr(n, s.astype(np.int32), d.astype(np.int32))
    h = hn.Hornet.from_csr(off, adj)
    ms = hn.BfsMulti(h)
    ms.set_params(0, alpha)
    srcs = rng.integers(0, n, 40).astype(np.int32)
    assert np.array_equal(ms.run(srcs).cpu().numpy(), expected(off, adj, srcs))


@pytest.mark.parametrize("limit", [1, 2, 14, 15, 16, 63])
def test_depth_limits(hn, limit):
    print("case msbfs limits", limit, flush=True)
    rows, cols = 9, 31
    i = np.arange(rows * cols, dtype=np.int32).reshape(rows, cols)
    s = np.concatenate([i[:, :-1].ravel(), i[:-1].ravel()])
    d = np.concatenate([i[:, 1:].ravel(), i[1:].ravel()])
    off, adj = O.coo_to_csr(rows * cols, s, d)
    h = hn.Hornet.from_csr(off, adj)
    ms = hn.BfsMulti(h)
    srcs = np.arange(0, 60, 3, dtype=np.int32)
    for limits in (np.full(srcs.size, limit), np.where(np.arange(srcs.size) % 3, limit, 0), np.zeros(srcs.size)):
        limits = limits.astype(np.int32)
        got = ms.run(srcs, depth_limits=limits).cpu().numpy()
        assert np.array_equal(got, expected(off, adj, srcs, limits))


@pytest.mark.parametrize("n", [1 << 20, (1 << 20) + 3])
def test_few_reached_of_many(hn, n):
    """Both sides of where the codes of unreached vertices are not read."""
    print("case msbfs few reached", n, flush=True)
    rng = np.random.default_rng(n)
    s, d = rng.integers(0, n, 3000).astype(np.int32), rng.integers(0, n, 3000).astype(np.int32)
    v = np.arange(n - 40, n - 1, dtype=np.int32)   # a path that ends in the last vertex
    off, adj = O.coo_to_csr(n, np.concatenate([s, v]), np.concatenate([d, v + 1]))
    h = hn.Hornet.from_csr(off, adj)
    srcs = np.concatenate([s[:15], v[:1], v[-1:]]).astype(np.int32)
    ms = hn.BfsMulti(h)
    for _ in range(2):
        assert np.array_equal(ms.run(srcs).cpu().numpy(), expected(off, adj, srcs))
