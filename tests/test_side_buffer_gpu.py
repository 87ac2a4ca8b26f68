"""Updates that defer more entries than the side buffer of a fresh handle holds, and
as many again once it does: rows that grow and shrink at their front, in place."""
import numpy as np
import pytest

from hornet_amd.graph import BatchUpdate, Hornet, HornetInit

pytestmark = pytest.mark.gpu


def check(h, rows, row_meta):
    out = h.getCOO(meta=row_meta is not None)
    n = [r.size for r in rows]
    assert np.array_equal(out[0].cpu().numpy(), np.repeat(np.arange(len(rows)), n))
    assert np.array_equal(out[1].cpu().numpy(), np.concatenate(rows))
    if row_meta is not None:
        assert np.array_equal(out[2][0].cpu().numpy(), np.concatenate(row_meta))


@pytest.mark.parametrize("nrows,meta", [(1, False), (24, False), (24, True)])
def test_front_of_long_rows(nrows, meta):
    print("case side buffer", nrows, meta, flush=True)
    nv, low, high = 40000, 1500, 30000
    old = np.arange(2000, 2000 + high, dtype=np.int32)   # blocks of 32,768 slots: 31,500 fit in place
    new = np.arange(low, dtype=np.int32)
    off = np.concatenate([np.arange(nrows + 1) * high, np.full(nv - nrows, nrows * high)]).astype(np.int32)
    init = HornetInit(nv, nrows * high, off, np.tile(old, nrows))
    f_old = np.arange(nrows * high, dtype=np.int32)
    h = Hornet(init.insertEdgeData(f_old) if meta else init)
    src = np.repeat(np.arange(nrows), low).astype(np.int32)
    dst = np.tile(new, nrows)
    f_new = -1 - np.arange(src.size, dtype=np.int32)
    empty = [np.zeros(0, np.int32)] * (nv - nrows)
    before = [old] * nrows + empty
    after = [np.concatenate([new, old])] * nrows + empty
    m_before = [f_old[i * high:(i + 1) * high] for i in range(nrows)] + empty if meta else None
    m_after = [np.concatenate([f_new[i * low:(i + 1) * low], f_old[i * high:(i + 1) * high]])
               for i in range(nrows)] + empty if meta else None
    for _ in range(2):
        assert h.insert(BatchUpdate(src, dst, meta=[f_new] if meta else None), True, True) == src.size
        check(h, after, m_after)
        assert h.erase(BatchUpdate(src, dst), True) == src.size
        check(h, before, m_before)
    assert h.update_stats()["applied"] == src.size
