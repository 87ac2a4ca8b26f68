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


@pytest.mark.parametrize("meta", [False, True])
def test_no_memory_for_the_entries(meta, monkeypatch):
    """A batch that is stopped because its deferred entries do not fit, and no memory for
    them: the graph and its blocks are as before, and the batch works later on."""
    from hornet_amd import HornetError
    print("case side buffer fails", meta, flush=True)
    nv, nrows, low, high = 40000, 24, 1500, 30000
    old, new = np.arange(2000, 2000 + high, dtype=np.int32), np.arange(low, dtype=np.int32)
    off = np.concatenate([np.arange(nrows + 1) * high, np.full(nv - nrows, nrows * high)]).astype(np.int32)
    init = HornetInit(nv, nrows * high, off, np.tile(old, nrows))
    f_old = np.arange(nrows * high, dtype=np.int32)
    h = Hornet(init.insertEdgeData(f_old) if meta else init)
    # rows at the front of long ones, and rows of their own, whose blocks are new
    src = np.concatenate([np.repeat(np.arange(nrows), low), np.arange(100, 200)]).astype(np.int32)
    dst = np.concatenate([np.tile(new, nrows), np.arange(100)]).astype(np.int32)
    f_new = -1 - np.arange(src.size, dtype=np.int32)
    batch = BatchUpdate(src, dst, meta=[f_new] if meta else None)
    before = [old] * nrows + [np.zeros(0, np.int32)] * (nv - nrows)
    own = [np.array([v - 100] if 100 <= v < 200 else [], np.int32) for v in range(nrows, nv)]
    after = [np.concatenate([new, old])] * nrows + own
    m_old = [f_old[i * high:(i + 1) * high] for i in range(nrows)]
    m_before = m_old + before[nrows:] if meta else None
    m_after = [np.concatenate([f_new[i * low:(i + 1) * low], m_old[i]]) for i in range(nrows)] + \
        [f_new[nrows * low + v - 100:][:1] if 100 <= v < 200 else np.zeros(0, np.int32) for v in range(nrows, nv)] if meta else None
    memory = h.memory()
    monkeypatch.setenv("HORNET_HIP_FAIL_SIDE_RESERVE", "2")
    for _ in range(2):
        with pytest.raises(HornetError):
            h.insert(batch, True, True)
        check(h, before, m_before)
        assert h.nE() == nrows * high and h.memory() == memory
    monkeypatch.delenv("HORNET_HIP_FAIL_SIDE_RESERVE")
    assert h.insert(batch, True, True) == src.size
    check(h, after, m_after)
    h2 = Hornet(HornetInit(nv, nrows * (low + high), (off.astype(np.int64) // high * (low + high)).astype(np.int32),
                           np.tile(np.concatenate([new, old]), nrows)))
    memory = h2.memory()
    gone = BatchUpdate(np.repeat(np.arange(nrows), low).astype(np.int32), np.tile(new, nrows))
    monkeypatch.setenv("HORNET_HIP_FAIL_SIDE_RESERVE", "2")
    with pytest.raises(HornetError):
        h2.erase(gone, True)
    check(h2, after[:nrows] + before[nrows:], None)
    assert h2.memory() == memory
    monkeypatch.delenv("HORNET_HIP_FAIL_SIDE_RESERVE")
    assert h2.erase(gone, True) == nrows * low
    check(h2, before, None)
