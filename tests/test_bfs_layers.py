"""BFS where most unreached vertices know no vertex of the frontier (layers): whether a
round pulls is decided by what the round before it discovered."""
import ctypes
import os
import random
import subprocess

import numpy as np
import pytest

import oracle as O

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hornet_amd", "csrc")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text('''#include "bfs_pulls.hpp"
extern "C" uint64_t quotient(uint64_t x, uint64_t d) { return hn::bfs_quotient(x, d); }
extern "C" uint64_t wasted(uint64_t size, uint32_t W, uint32_t prev, uint64_t open, uint64_t mu) { return hn::bfs_wasted(size, W, prev, open, mu); }
extern "C" bool rule(uint64_t size, uint32_t W, uint64_t scan, uint64_t vis, int64_t nv, int64_t ne, uint32_t prev) { return hn::bfs_pulls(size, W, scan, vis, nv, ne, prev); }
''')
    out = []
    for i, flags in enumerate((["-O0", "-fsanitize=undefined", "-fno-sanitize-recover"], ["-O3", "-mfma", "-ffp-contract=fast"])):
        so = str(d / f"rule{i}.so")
        subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", *flags, f"-I{CSRC}", str(d / "rule.cpp"), "-o", so], check=True)
        lib = ctypes.CDLL(so)
        u32, u64, i64 = ctypes.c_uint32, ctypes.c_uint64, ctypes.c_int64
        lib.quotient.restype = lib.wasted.restype = u64
        lib.quotient.argtypes = [u64, u64]
        lib.wasted.argtypes = [u64, u32, u32, u64, u64]
        lib.rule.restype = ctypes.c_bool
        lib.rule.argtypes = [u64, u32, u64, u64, i64, i64, u32]
        out.append(lib)
    return out


def test_quotient(rules):
    rng = random.Random(1)
    pairs = [(0, 1), (1, 1), (2**63 - 1, 1), (2**63 - 1, 2**32 - 1), (2**63 - 1, 2**31)]
    pairs += [(int(2 ** rng.uniform(0, 63)), int(2 ** rng.uniform(0, 32))) for _ in range(3000)]
    for x, d in pairs:
        got = {r.quotient(x, d) for r in rules}
        assert len(got) == 1
        q = got.pop()
        if x // d < 2**47:   # (beyond, only that it is large matters)
            assert abs(q - x / d) <= 0.04 * x / d + 2, (x, d, q)
        else:
            assert q > 2**46


def test_compiled_alike_at_the_limits(rules):
    """No overflow (the sanitizer's build), and one answer however it is compiled."""
    rng = random.Random(2)
    for _ in range(5000):
        nv = int(2 ** rng.uniform(1, 31))
        ne = min(int(nv * 2 ** rng.uniform(-1, 8)), 2**32 - 2)
        scan, vis = rng.choice([0, rng.randrange(ne + 1), ne]), rng.randrange(nv)
        size = rng.choice([1, rng.randrange(1, nv - vis + 1), nv - vis])
        W, prev = (rng.choice([1, 4097, rng.randrange(1, 2**32), 2**32 - 1]) for _ in range(2))
        args = (size, W, scan, vis, nv, ne, rng.choice([0, prev]))
        assert len({r.rule(*args) for r in rules}) == 1, args
        args = (size, W, prev, nv - vis - size, max(ne - scan, 0))
        assert len({r.wasted(*args) for r in rules}) == 1, args


@pytest.mark.parametrize("size,W,scan,vis,nv,ne,prev,want", [
    # a layer of twenty, 16 edges a vertex to the next one: the frontier reaches one layer of the others
    (600, 4970, 100_000, 4000, 12000, 360170, 9594, False),
    (2000, 16700, 300_000, 16000, 40000, 1211424, 16675, False),
    (20000, 167440, 4_000_000, 200000, 400000, 12155532, 167463, False),
    # R-MAT: a hub's neighbours, and what those reach
    (64370, 5513142, 64_000, 1, 1048576, 31402126, 16093, True),
    (541559, 2575151, 22_000_000, 64371, 1048576, 31402126, 5513142, True),
    # uniform random
    (65839, 304065, 80_000, 4548, 1048576, 16777068, 19733, True),
    # nothing known of the frontier before: as without it
    (600, 4970, 100_000, 4000, 12000, 360170, 0, True),
])
def test_layers_push_and_others_pull(rules, size, W, scan, vis, nv, ne, prev, want):
    assert [r.rule(size, W, scan, vis, nv, ne, prev) for r in rules] == [want] * 2


def check(h, off, adj, source):
    import torch

    import hornet_amd.graph as G
    bfs = G.BfsTopDown(h)
    bfs.set_parameters(source)
    want, levels = O.bfs(off, adj, source)
    for _ in range(2):
        bfs.d_distances.fill_(-7)
        bfs.run()
        assert np.array_equal(bfs.distances().cpu().numpy(), want)
    torch.cuda.synchronize()
    assert bfs.stats.visited == int((want != G.INF).sum())


@pytest.mark.gpu
@pytest.mark.parametrize("k,w,deg", [(20, 300, 16), (20, 600, 16), (20, 600, 64), (20, 2000, 64), (20, 20000, 16)])
def test_layers(k, w, deg):
    """From the first layer, the last, and the middle: pulls at first, then pushes, then pulls."""
    import torch

    import hornet_amd.graph as G
    print(f"case layers {k} {w} {deg}", flush=True)
    rng = np.random.default_rng(w + deg)
    u = np.repeat(np.arange((k - 1) * w), deg)
    v = (u // w + 1) * w + rng.integers(0, w, u.size)
    h = G.Hornet.from_coo_device(k * w, *(torch.from_numpy(x.astype(np.int32)).cuda() for x in (u, v)))
    off, adj = (x.cpu().numpy() for x in h.getCSR())
    for source in (0, k * w - 1, k // 2 * w):
        check(h, off, adj, source)


@pytest.mark.gpu
@pytest.mark.parametrize("nv", [8193, 65504, 65535, 65536, 65537, 65600])
def test_pull_spans(nv):
    """Graphs on both sides of where a wave pulls for 64 vertices instead of 256."""
    import torch

    import hornet_amd.graph as G
    print(f"case pull spans {nv}", flush=True)
    rng = np.random.default_rng(nv)
    s, d = rng.integers(0, nv, (2, 8 * nv))
    h = G.Hornet.from_coo_device(nv, *(torch.from_numpy(x.astype(np.int32)).cuda() for x in (s, d)))
    off, adj = (x.cpu().numpy() for x in h.getCSR())
    check(h, off, adj, 0)
    check(h, off, adj, nv - 1)
