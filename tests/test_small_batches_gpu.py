"""Batches around the sizes up to which one workgroup sorts and scans them."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hn():
    import hornet_amd.graph as G
    return G


def coo(off, adj):
    return np.repeat(np.arange(off.size - 1), np.diff(off)).astype(np.int32), adj.astype(np.int32)


def check_equal(h, off, adj):
    s, d = h.getCOO()
    xs, xd = coo(off, adj)
    assert np.array_equal(s.cpu().numpy(), xs) and np.array_equal(d.cpu().numpy(), xd)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1024, 1025, 4097, 8191, 8192, 8193, 16385])
@pytest.mark.parametrize("dedup", [False, True])
def test_insert_and_erase(hn, n, dedup):
    print("case small batch", n, dedup, flush=True)
    off, adj = O.rmat_graph(12, seed=5)
    h = hn.Hornet.from_csr(off, adj)
    nv = off.size - 1
    rng = np.random.default_rng(n)
    # a few sources with long runs of equal keys beside uniform ones, both ends of the id range
    bs = np.where(rng.random(n) < 0.3, rng.choice([0, 7, nv - 1], n), rng.integers(0, nv, n)).astype(np.int32)
    bd = np.where(rng.random(n) < 0.3, rng.choice([0, 5, nv - 1], n), rng.integers(0, nv, n)).astype(np.int32)
    got = h.insert(hn.BatchUpdate(bs, bd), dedup, dedup)
    o2, a2, added = O.insert(off, adj, bs, bd, dedup, dedup)
    assert got == added
    check_equal(h, o2, a2)
    got = h.erase(hn.BatchUpdate(bs, bd), True)
    o3, a3, removed = O.erase(o2, a2, bs, bd, True)
    assert got == removed
    check_equal(h, o3, a3)


@pytest.mark.parametrize("n", [1, 64, 1025, 8192, 8193])
def test_fields_keep_the_order_of_equal_pairs(hn, n):
    print("case small batch fields", n, flush=True)
    off = np.zeros(101, dtype=np.int64)
    h = hn.Hornet(hn.HornetInit(100, 0, off, np.zeros(0, np.int32)).insertEdgeData(np.zeros(0, np.int32)))
    rng = np.random.default_rng(n)
    bs, bd = rng.integers(0, 100, n).astype(np.int32), rng.integers(0, 9, n).astype(np.int32)
    f = np.arange(n, dtype=np.int32)
    h.insert(hn.BatchUpdate(bs, bd, meta=[f]))
    s, d, m = h.getCOO(meta=True)
    order = np.lexsort((f, bd, bs))
    assert np.array_equal(s.cpu().numpy(), bs[order]) and np.array_equal(d.cpu().numpy(), bd[order])
    assert np.array_equal(m[0].cpu().numpy(), f[order])


@pytest.mark.parametrize("scale", [10, 19])
@pytest.mark.parametrize("n", [100, 4095, 4096])
def test_there_and_back(hn, scale, n):
    """Gaps of an erase on both sides of one workgroup's scan, and copy tiles
    (s19: 15 M entries) that are too many for one where the batch is not."""
    import torch
    print("case small batch there and back", scale, n, flush=True)
    h = hn.Hornet.rmat(scale, 3, edge_factor=16)
    off, adj = (x.clone() for x in h.getCSR())
    rng = np.random.default_rng(n)
    v = 1 << scale
    s = torch.from_numpy(rng.integers(0, v, n).astype(np.int32)).cuda()
    d = torch.from_numpy(rng.integers(0, v, n).astype(np.int32)).cuda()
    src = torch.repeat_interleave(torch.arange(v, device="cuda"), off[1:] - off[:-1])
    old = src * v + adj
    new = torch.unique(s.long() * v + d)
    both = torch.unique(torch.cat([old, new]))
    h.insert(hn.BatchUpdate(s, d), True, True)
    cs, cd = h.getCOO()
    assert torch.equal(cs.long() * v + cd, both)
    h.erase(hn.BatchUpdate(s, d), True)
    cs, cd = h.getCOO()
    assert torch.equal(cs.long() * v + cd, old[~torch.isin(old, new)])
