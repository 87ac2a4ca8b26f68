"""Triangle counts of graphs whose vertices have almost all no entries: the passes over
vertices go by bits, 64 to a word and four words to a wave, and lists of 2 to 16
entries and of more have bits of their own."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nv", [63, 64, 65, 257, 65535, 70001, (1 << 20) - 255, (1 << 20) + 1])
@pytest.mark.parametrize("stored", [False, True])
def test_few_entries(nv, stored):
    """Cliques with lists of 1 to 17 entries (oriented; 2, 16 and 17 as stored) at the
    first vertices, the last, and across a word and four of them."""
    import torch

    import hornet_amd.graph as G
    print(f"case tc sparse nv={nv} stored={stored}", flush=True)
    at = [(0, 3), (3, 17), (nv - 18, 18)] + ([(64 * k - 9, 18) for k in (2, 3, nv // 128)] if nv > 256 else [])
    src, dst = (torch.from_numpy(np.concatenate([v + np.triu_indices(n, 1)[e] for v, n in at]).astype(np.int32)).cuda()
                for e in (0, 1))
    h = G.Hornet.from_coo_device(nv, src, dst)
    off, adj = (x.cpu().numpy() for x in h.getCSR())
    tc = G.TriangleCounting2(h)
    tc.init()
    want = O.tc2_per_vertex(*((off, adj) if stored else O.directed_by_degree(off, adj)))
    for _ in range(2):   # the second one on dirty scratch
        (tc.run if stored else tc.run_undirected)()
        assert tc.countTriangles() == int(want.sum()) and np.array_equal(tc.copyTCToHost(), want)


@pytest.mark.parametrize("length", [16, 17, 600])
def test_edges_grouped_in_some_tiles(length):
    """Stored rows of four entries, of which those of every sixteenth thousand vertices
    also go to one of three long lists: most tiles of rows hold no edge that its
    destination owns."""
    import torch

    import hornet_amd.graph as G
    print(f"case tc grouped tiles length={length}", flush=True)
    nv, rng = 100_003, np.random.default_rng(length)
    src = np.repeat(np.arange(nv), 4)
    dst = rng.integers(0, 2000, src.size)
    some = np.flatnonzero(np.arange(nv) // 1000 % 16 == 3)
    long = np.array([5, 50_000, nv - 1])
    src = np.concatenate([src, np.repeat(some, 3), np.repeat(long, length - 4)])
    dst = np.concatenate([dst, np.tile(long, some.size), rng.integers(0, 2000, 3 * (length - 4))])
    k = np.unique(src * nv + dst)
    src, dst = (torch.from_numpy(x.astype(np.int32)).cuda() for x in (k // nv, k % nv))
    h = G.Hornet.from_coo_device(nv, src, dst, symmetrize=False, drop_self_loops=False)
    want = O.tc2_per_vertex(*(x.cpu().numpy() for x in h.getCSR()))
    assert want.any()
    tc = G.TriangleCounting2(h)
    tc.init()
    for _ in range(2):
        tc.run()
        assert tc.countTriangles() == int(want.sum()) and np.array_equal(tc.copyTCToHost(), want)


@pytest.mark.parametrize("nv", [65535, 65536])
@pytest.mark.parametrize("stored", [False, True])
def test_lists_around_the_small_ones(nv, stored):
    """Cliques whose lists have 15 to 18 and 30 to 34 entries, stored as they are and from a
    CSR (not known to be symmetric), on both sides of where lists of 32 count as short."""
    import torch

    import hornet_amd.graph as G
    print(f"case tc short lists nv={nv} stored={stored}", flush=True)
    sizes = [16, 17, 18, 19, 31, 32, 33, 34, 35] * 2
    at = np.cumsum([0] + [n + 7 for n in sizes])
    src, dst = (np.concatenate([v + np.triu_indices(n, 1)[e] for v, n in zip(at, sizes)]) for e in (0, 1))
    # and edges between lists of different lengths
    rng = np.random.default_rng(5)
    more = rng.integers(0, at[-1], (2, 400))
    src, dst = np.concatenate([src, more[0]]), np.concatenate([dst, more[1]])
    h = G.Hornet.from_coo_device(nv, *(torch.from_numpy(x.astype(np.int32)).cuda() for x in (src, dst)))
    h = G.Hornet.from_device_csr(*h.getCSR())
    off, adj = (x.cpu().numpy() for x in h.getCSR())
    want = O.tc2_per_vertex(*((off, adj) if stored else O.directed_by_degree(off, adj)))
    tc = G.TriangleCounting2(h)
    tc.init()
    for _ in range(2):
        (tc.run if stored else tc.run_undirected)()
        assert tc.countTriangles() == int(want.sum()) and np.array_equal(tc.copyTCToHost(), want)
