"""BFS where whole-device rounds write distances themselves: from 126 on they do not fit
the state bytes, and only the one-workgroup levels of long thin graphs meet that
otherwise.  And graphs of more than 2^25 vertices, whose pulls go without the summary of
visited vertices.  Layered graphs, whose distances are the layers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
INF = 2**31 - 1


@pytest.fixture(scope="module")
def hn():
    import hornet_amd.graph as G
    return G


def layered(hn, sizes, fan, directed, lone=5, seed=1):
    """Every vertex of a layer has `fan` neighbours in the layer before; ids are permuted;
    `lone` vertices have none.  The graph, the source and every vertex's distance."""
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    first = np.concatenate([[0], np.cumsum(sizes)])
    n = int(first[-1]) + lone
    name = torch.randperm(n, device="cuda", generator=g, dtype=torch.int32)
    src, dst = [], []
    for k in range(1, len(sizes)):
        v = torch.arange(int(first[k]), int(first[k + 1]), device="cuda")
        for _ in range(min(fan, int(sizes[k - 1]))):
            # (every vertex of the layer before has a part in it)
            up = (v + torch.randint(0, 1 << 30, (1,), device="cuda", generator=g)) % int(sizes[k - 1]) + int(first[k - 1])
            src.append(name[up]), dst.append(name[v])
    h = hn.Hornet.from_coo_device(n, torch.cat(src), torch.cat(dst), symmetrize=not directed)
    dist = torch.full((n,), INF, dtype=torch.int32, device="cuda")
    for k in range(len(sizes)):
        dist[name[int(first[k]):int(first[k + 1])].long()] = k
    return h, int(name[0]), dist


def check(hn, h, source, dist):
    import torch
    bfs = hn.BfsTopDown(h)
    bfs.set_parameters(source)
    for poison in (-7, 12345):   # the second one queues as many rounds as the first needed
        bfs.d_distances.fill_(poison)
        bfs.run()
        wrong = torch.nonzero(bfs.distances() != dist).flatten()
        assert wrong.numel() == 0, (wrong[:5], bfs.distances()[wrong[:5]], dist[wrong[:5]])
    assert bfs.stats.levels == int(dist[dist != INF].max()) + 1
    assert bfs.stats.visited == int((dist != INF).sum())


# layers that a round pushes, of 30,000 and 400,000 vertices, and that it pulls (where
# storage is known to be symmetric), at distances on both sides of 125 and 126
@pytest.mark.parametrize("directed", [False, True])
@pytest.mark.parametrize("path", [119, 121, 122, 123, 124, 125, 126, 127, 130])
def test_wide_levels_far_from_the_source(hn, path, directed):
    print(f"case bfs deep path={path} directed={directed}", flush=True)
    sizes = [1] * path + [500, 30011, 400000, 400003, 29000, 600, 1, 1]
    check(hn, *layered(hn, sizes, 3, directed))


@pytest.mark.parametrize("path", [1, 124])
def test_more_than_2_25_vertices(hn, path):
    print(f"case bfs big path={path}", flush=True)
    sizes = [1] * path + [1000, 3001, 1 << 20, 1 << 25, 70000, 3, 1]
    check(hn, *layered(hn, sizes, 2, False, lone=77))


# bitmap in LDS and in memory; a bit of the summary stands for 128 vertices up to 2^24, then for 256
@pytest.mark.parametrize("rest", [600000, 1 << 20, (1 << 24) - 52000, (1 << 24) + 77, 20000003])
def test_summary_of_visited_vertices(hn, rest):
    """Levels by one workgroup, then a pull that asks the summary they have written: few
    vertices are visited and their rows hold most entries."""
    print(f"case bfs summary rest={rest}", flush=True)
    check(hn, *layered(hn, [1, 1, 1, 200, 900, 50000, rest, 3, 1], 2, False))


# the frontier doubles on ids that share words of the bitmap and of the summary
@pytest.mark.parametrize("directed", [False, True])
@pytest.mark.parametrize("n", [3000, 700001, (1 << 20) - 1, 2000003])
def test_binary_trees(hn, n, directed):
    import torch
    print(f"case bfs tree n={n} directed={directed}", flush=True)
    v = torch.arange(1, n, dtype=torch.int32, device="cuda")
    h = hn.Hornet.from_coo_device(n + 3, (v - 1) // 2, v, symmetrize=not directed)
    dist = torch.full((n + 3,), INF, dtype=torch.int32, device="cuda")
    dist[:n] = torch.from_numpy(np.frexp(np.arange(1, n + 1))[1] - 1).to(dist)
    check(hn, h, 0, dist)
