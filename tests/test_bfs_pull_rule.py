"""Push or pull is decided by several kernels on their own, which must agree: the rule
is the same to the last bit however it is compiled."""
import ctypes
import os
import random
import subprocess
from fractions import Fraction

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hornet_amd", "csrc")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    """The rule with and without contracted products, optimised and not."""
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text('#include "bfs_pulls.hpp"\nextern "C" bool rule(uint64_t size, uint32_t W, uint64_t scan, '
                                'uint64_t vis, int64_t nv, int64_t ne) { return hn::bfs_pulls(size, W, scan, vis, nv, ne); }\n')
    out = []
    for i, flags in enumerate((["-O0"], ["-O3", "-mfma", "-ffp-contract=fast"], ["-O3", "-ffp-contract=off"])):
        so = str(d / f"rule{i}.so")
        subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", *flags, f"-I{CSRC}", str(d / "rule.cpp"), "-o", so], check=True)
        f = ctypes.CDLL(so).rule
        f.restype = ctypes.c_bool
        f.argtypes = [ctypes.c_uint64, ctypes.c_uint32, ctypes.c_uint64, ctypes.c_uint64, ctypes.c_int64, ctypes.c_int64]
        out.append(f)
    return out


def exact(size, W, scan, vis, nv, ne):
    if W <= 4096:
        return False
    mf = 4 * W
    mu = max(ne - scan - mf, 0)
    touch = min(nv - vis - size, mu)
    slots = min(Fraction(mu), Fraction(touch * ne, mf))
    return 4 * nv + 16 * touch + slots / 2 < 7 * mf + 20 * min(mf, touch)


def test_every_copy_agrees(rules):
    rng = random.Random(7)
    pulls = 0
    for _ in range(4000):
        nv = int(2 ** rng.uniform(13, 31)) - rng.randrange(2)
        ne = min(int(nv * 2 ** rng.uniform(-1, 6)), 2**32 - 2)
        scan, vis = rng.randrange(ne + 1), rng.randrange(nv)
        size = rng.randrange(1, nv - vis + 1)
        lo, hi = 4097, max(4098, min(ne, 2**32 - 1))
        near = [lo, hi, rng.randrange(lo, hi + 1)]
        # and the frontiers where the rule turns over
        if exact(size, lo, scan, vis, nv, ne) != exact(size, hi, scan, vis, nv, ne):
            while hi - lo > 1:
                mid = (lo + hi) // 2
                if exact(size, mid, scan, vis, nv, ne) == exact(size, hi, scan, vis, nv, ne):
                    hi = mid
                else:
                    lo = mid
            near += [lo - 1, lo, hi, hi + 1]
        for W in near:
            W = min(W, 2**32 - 1)
            want = exact(size, W, scan, vis, nv, ne)
            pulls += want
            assert [f(size, W, scan, vis, nv, ne) for f in rules] == [want] * 3, (size, W, scan, vis, nv, ne)
    assert pulls > 1000


@pytest.mark.parametrize("W", [0, 1, 4095, 4096])
def test_small_frontiers_push(rules, W):
    assert not any(f(4096, W, 0, 0, 10**6, 10**8) for f in rules)
