"""Sorts at the sizes where the tiles of a pass change: builds from an edge list
(keys alone) and from unsorted rows with a field (keys with positions)."""
import numpy as np
import pytest
import torch

from hornet_amd.graph import Hornet, HornetInit

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [16383, 16384, 16385, (1 << 20) - 1, 1 << 20, (1 << 23) - 1, (1 << 23) + 4097])
def test_build_from_pairs(m):
    print("case sort tiles", m, flush=True)
    n = 99991
    rng = np.random.default_rng(m)
    # long runs of equal digits beside uniform ones
    s = np.where(rng.random(m) < 0.2, 4711, rng.integers(0, n, m)).astype(np.int32)
    d = np.where(rng.random(m) < 0.2, rng.integers(0, 300, m), rng.integers(0, n, m)).astype(np.int32)
    h = Hornet.from_coo_device(n, torch.from_numpy(s).cuda(), torch.from_numpy(d).cuda(), symmetrize=False,
                               drop_self_loops=False)
    key = np.unique(s.astype(np.int64) * n + d)
    gs, gd = h.getCOO()
    assert np.array_equal(gs.cpu().numpy().astype(np.int64) * n + gd.cpu().numpy(), key)


@pytest.mark.parametrize("m", [8192, 8193, 16385, (1 << 20) + 1])
def test_rows_with_a_field(m):
    print("case sort tiles field", m, flush=True)
    n = 5003
    rng = np.random.default_rng(m)
    s = np.sort(rng.integers(0, n, m))
    d = rng.integers(0, n, m).astype(np.int32)
    off = np.concatenate([[0], np.cumsum(np.bincount(s, minlength=n))]).astype(np.int32)
    f = np.arange(m, dtype=np.int32)
    h = Hornet(HornetInit(n, m, off, d).insertEdgeData(f))
    order = np.lexsort((f, d, s))
    gs, gd, meta = h.getCOO(meta=True)
    assert np.array_equal(gs.cpu().numpy(), s[order]) and np.array_equal(gd.cpu().numpy(), d[order])
    assert np.array_equal(meta[0].cpu().numpy(), f[order])


@pytest.mark.parametrize("m", [(1 << 20) - 1, 1 << 20, (1 << 23) - 1])
def test_batches(m):
    """An update lays its scratch out for one key more than it sorts."""
    print("case sort tiles batch", m, flush=True)
    n = 4099
    rng = np.random.default_rng(m)
    s, d = rng.integers(0, n, m).astype(np.int32), rng.integers(0, n, m).astype(np.int32)
    h = Hornet(HornetInit(n, 0, np.zeros(n + 1, np.int32), np.zeros(0, np.int32)))
    from hornet_amd.graph import BatchUpdate
    key = np.unique(s.astype(np.int64) * n + d)
    assert h.insert(BatchUpdate(s, d), True, True) == key.size
    gs, gd = h.getCOO()
    assert np.array_equal(gs.cpu().numpy().astype(np.int64) * n + gd.cpu().numpy(), key)
    assert h.erase(BatchUpdate(s, d), True) == key.size and h.nE() == 0
