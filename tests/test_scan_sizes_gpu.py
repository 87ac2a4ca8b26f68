"""Vertex counts on both sides of the scans' forms: one workgroup, small tiles, large ones."""
import numpy as np
import pytest

from hornet_amd.graph import Hornet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nv", [1, 1023, 1024, 8191, 8192, 8193, 9217, (1 << 22) - 1, 1 << 22, (1 << 22) + 1, 4300801])
def test_offsets(nv):
    print("case scan sizes", nv, flush=True)
    rng = np.random.default_rng(nv)
    rows = np.unique(np.concatenate([[0, nv - 1], rng.integers(0, nv, 4000)]))
    deg = np.zeros(nv, dtype=np.int64)
    deg[rows] = rng.integers(1, 4, rows.size)
    deg = np.minimum(deg, nv)
    off = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    adj = (np.arange(off[-1]) - np.repeat(off[:-1], deg)).astype(np.int32)   # 0, 1, .. in every row
    o, e = Hornet.from_csr(off, adj).getCSR()
    assert np.array_equal(o.cpu().numpy(), off) and np.array_equal(e.cpu().numpy(), adj)
