"""Edge lists to rows where tiles of 4,096 sorted keys and their waves end: repeats
across every border, one pair only, nothing left, first and last vertices without rows."""
import numpy as np
import pytest
import torch

from hornet_amd.graph import Hornet

pytestmark = pytest.mark.gpu


def build(n, s, d, **kw):
    return Hornet.from_coo_device(n, torch.from_numpy(s.astype(np.int32)).cuda(),
                                  torch.from_numpy(d.astype(np.int32)).cuda(), **kw)


def check(h, n, s, d):
    key = np.unique(s.astype(np.int64) * n + d)
    off, adj = h.getCSR()
    assert np.array_equal(adj.cpu().numpy(), (key % n).astype(np.int32))
    assert np.array_equal(off.cpu().numpy(), np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))]))


@pytest.mark.parametrize("m", [1, 63, 64, 65, 1023, 1024, 1025, 4095, 4096, 4097, 8192, 20481])
@pytest.mark.parametrize("spread", [1, 3, 700, 1 << 20])
def test_rows(m, spread):
    print("case unique rows", m, spread, flush=True)
    n = 5003
    rng = np.random.default_rng(m * 31 + spread)
    s = 17 + rng.integers(0, min(spread, n - 40), m)   # ends of the id range without rows
    d = rng.integers(0, min(spread, n), m)
    check(build(n, s, d, symmetrize=False, drop_self_loops=False), n, s, d)


@pytest.mark.parametrize("m", [1, 4096, 5000])
def test_one_pair_and_none(m):
    print("case unique rows ends", m, flush=True)
    for n, a, b in ((8, 7, 7), (8, 0, 7), (9, 8, 0), (1, 0, 0)):
        s, d = np.full(m, a), np.full(m, b)
        check(build(n, s, d, symmetrize=False, drop_self_loops=False), n, s, d)
    h = build(5, np.arange(m) % 5, np.arange(m) % 5)   # loops only: dropped
    assert h.nE() == 0 and not h.getCSR()[0].cpu().numpy().any()
