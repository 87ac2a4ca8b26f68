"""Build and export move entries in tiles of 2,048 whose segments are staged, or
searched where more than 8,192 lie in one tile: rows and empty rows at those limits."""
import numpy as np
import pytest

from hornet_amd.graph import Hornet, HornetInit

pytestmark = pytest.mark.gpu

DEGREES = {
    "one": [1],
    "empty_ends": [0, 0, 3, 0],
    "tile_less": [2047],
    "tile": [2048],
    "tile_more": [2049, 1],
    "rows_of_one": [1] * 4099,
    "around_four": [1, 2, 3, 4, 5, 6, 7, 8, 9] * 300,
    "long_and_short": [5000, 1, 0, 0, 2, 4095, 3],
    "staged_limit": [1] + [0] * 8189 + [1],          # (with the row after it) 8,192 segments in the one tile
    "past_the_limit": [1] + [0] * 8190 + [2, 5],
    "far_past": [3] + [0] * 70001 + [2500] + [0] * 300 + [7],
    "more_than_block": ([0, 1] * 700 + [9]) * 3,
}


@pytest.mark.parametrize("name", DEGREES)
@pytest.mark.parametrize("meta", [False, True])
def test_rows_and_export(name, meta):
    print("case copy tiles", name, meta, flush=True)
    deg = np.array(DEGREES[name], dtype=np.int64)
    rng = np.random.default_rng(7)
    off = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    nv = max(deg.size, int(deg.max()) + 1)
    off = np.concatenate([off, np.full(nv - deg.size, off[-1], dtype=np.int32)])
    adj = np.concatenate([np.sort(rng.choice(nv, d, replace=False)) for d in deg]).astype(np.int32)
    fields = [rng.integers(-2**31, 2**31, adj.size).astype(np.int32),
              rng.integers(0, 2**63, adj.size, dtype=np.int64)] if meta else []
    init = HornetInit(nv, adj.size, off, adj)
    h = Hornet(init.insertEdgeData(*fields) if meta else init)
    o, e = h.getCSR()
    assert np.array_equal(o.cpu().numpy(), off) and np.array_equal(e.cpu().numpy(), adj)
    out = h.getCOO(meta=meta)
    assert np.array_equal(out[0].cpu().numpy(), np.repeat(np.arange(nv), np.diff(off)))
    assert np.array_equal(out[1].cpu().numpy(), adj)
    for got, exp in zip(out[2] if meta else [], fields):
        assert np.array_equal(got.cpu().numpy(), exp.view(got.cpu().numpy().dtype))
