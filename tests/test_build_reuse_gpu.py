"""Builds whose buffers are blocks that earlier handles gave back: sizes repeat and
change, from one thread and from several, each on its own stream."""
import threading

import numpy as np
import pytest
import torch

import oracle as O
from hornet_amd.graph import BatchUpdate, Hornet

pytestmark = pytest.mark.gpu

SIZES = [(10, 1), (13, 2), (10, 3), (0, 0), (12, 4), (13, 5), (10, 1)]


def work(errors, turn):
    try:
        with torch.cuda.stream(torch.cuda.Stream()):
            for k in range(2 * len(SIZES)):
                scale, seed = SIZES[(k + turn) % len(SIZES)]
                if scale == 0:
                    off, adj = np.zeros(2, dtype=np.int64), np.zeros(0, dtype=np.int32)
                else:
                    off, adj = O.rmat_graph(scale, seed=seed)
                h = Hornet.from_csr(off, adj)
                o, e = h.getCSR()
                assert np.array_equal(o.cpu().numpy(), off) and np.array_equal(e.cpu().numpy(), adj)
                if scale:
                    s = np.repeat(np.arange(off.size - 1), np.diff(off)).astype(np.int32)
                    assert h.erase(BatchUpdate(torch.from_numpy(s).cuda(), torch.from_numpy(adj).cuda())) == adj.size
                    assert h.nE() == 0
                h.release()
    except Exception as e:   # reported by the test's own thread
        errors.append(repr(e))


@pytest.mark.parametrize("threads", [1, 4])
def test_rebuild(threads):
    print("case build reuse", threads, flush=True)
    errors = []
    pool = [threading.Thread(target=work, args=(errors, i)) for i in range(threads)]
    for t in pool:
        t.start()
    for t in pool:
        t.join()
    assert not errors, errors


def test_what_is_kept_is_bounded():
    print("case build reuse bound", flush=True)
    torch.cuda.synchronize()
    before, _ = torch.cuda.mem_get_info()
    for scale in range(16, 21):
        Hornet.rmat(scale, seed=1, slack=1.0 + scale / 8).release()
    kept = before - torch.cuda.mem_get_info()[0]
    assert kept <= (5 << 30), kept   # 4 GiB, and what the driver rounds
