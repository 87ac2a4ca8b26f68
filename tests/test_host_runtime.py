"""The library's host side over a HIP runtime without a device (tests/cpp/fake_hip.cpp):
which buffers a captured launch names, what is waited for before memory is kept for
reuse, and what is given back.  Each test is a program of its own, as the runtime is
replaced for its whole process."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = r"""
import ctypes, sys
from ctypes import byref, c_bool, c_char_p, c_int32, c_int64, c_long, c_uint64, c_uint8, c_void_p
fake = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
fake.fake_trace.restype = c_char_p
fake.fake_used.restype = fake.fake_stale.restype = c_long
fake.fake_fail_after.argtypes = fake.fake_device_total.argtypes = [c_long]
lib.hn_last_error.restype = c_char_p
lib.hn_graph_create_csr.argtypes = [c_int32, c_int64, c_void_p, c_void_p, c_int32, ctypes.c_double, c_void_p, c_void_p]
lib.hn_graph_destroy.argtypes = [c_void_p]

def ok(status):
    assert status == 0, (status, lib.hn_last_error())

def graph(nv=1000):
    h = c_void_p()
    ok(lib.hn_graph_create_csr(nv, 0, (c_int64 * (nv + 1))(), (c_int32 * 1)(), 1, 0.0, None, byref(h)))
    return h
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "cpp", "fake_hip.cpp"), "-o", so, "-ldl"], check=True)
    return so


def program(fake, code):
    r = subprocess.run([sys.executable, "-c", PRELUDE + code, fake, os.path.join(ROOT, "hornet_amd", "libhornet_hip.so")],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def test_window_steps_follow_their_buffers(fake):
    """A window that fails after its keys' buffer has moved, a batch without a window,
    and a window again: what the captured window step names is allocated."""
    program(fake, r"""
m = {n: getattr(lib, "_ZN2hn" + n) for n in ("16ms_engine_createEP8hn_graphPPNS_8MsEngineE",
     "15ms_window_beginEPNS_8MsEngineEPKiS3_PKhlP12ihipStream_tPb", "13ms_window_endEPNS_8MsEngineEimPKmP12ihipStream_t",
     "15ms_window_clearEPNS_8MsEngineEP12ihipStream_t",
     "13ms_run_engineEPNS_8MsEngineEPKiiS3_PiP14hn_msbfs_statsP12ihipStream_t")}
create, begin, end, clear, run = m.values()
create.argtypes = [c_void_p, c_void_p]
begin.argtypes = [c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_void_p, c_void_p]
end.argtypes = [c_void_p, c_int32, c_uint64, c_void_p, c_void_p]
clear.argtypes = [c_void_p, c_void_p]
run.argtypes = [c_void_p, c_void_p, c_int32, c_void_p, c_void_p, c_void_p, c_void_p]
g, e = graph(), c_void_p()
sv = (c_uint64 * 64)()

def window(n, fail_after=-1):
    pairs, tags, sym = (c_int32 * n)(), (c_uint8 * n)(), c_bool()
    ok(begin(e, pairs, pairs, tags, n, None, byref(sym)))
    fake.fake_fail_after(fail_after)
    s = end(e, 1, 0, sv, None)
    fake.fake_fail_after(-1)
    if s == 0: batch()
    ok(clear(e, None))
    return s

def batch():
    ok(run(e, (c_int32 * 4)(1, 2, 3, 4), 4, None, None, None, None))

for k in range(8):                    # one reservation further each time
    ok(create(g, byref(e)))
    assert window(10) == 0
    assert (window(5000, k) != 0) == (k < 4), k          # four buffers grow with the window
    batch()                           # the step without a window is captured after that
    assert window(5000) == 0
    batch()
    assert window(10) == 0
    assert fake.fake_stale() == 0, (k, fake.fake_stale())
""")


@pytest.mark.parametrize("current", [0, 1])
def test_destroy_waits_for_the_graphs_device(fake, current):
    """Freed blocks are kept for reuse: the wait before that is for the device that they
    are on, whichever is current."""
    program(fake, f"current = {current}" + r"""
fake.hipSetDevice(1)
g = graph()
fake.hipSetDevice(current)
fake.fake_clear_trace()
ok(lib.hn_graph_destroy(g))
assert fake.fake_trace() == b"wait@1 ", fake.fake_trace()   # and nothing went back to the driver
d = c_int32(-1)
fake.hipGetDevice(byref(d))
assert d.value == current
""")


def test_memory_of_destroyed_graphs_is_given_back(fake):
    program(fake, r"""
base = fake.fake_used()
ok(lib.hn_graph_destroy(graph()))
assert fake.fake_used() > base            # kept for the next graph
ok(lib.hn_memory_trim())
assert fake.fake_used() == base
""")


def test_triangle_scratch_of_sparse_graphs(fake):
    """What a count reserves for vertices without entries: 40 bytes each, and a quarter
    more in a scratch buffer, in blocks that are rounded up by an eighth at most."""
    program(fake, r"""
nv = 1 << 20
off = (c_int64 * (nv + 1))(*([0, 1] + [2] * (nv - 1)))
h = c_void_p()
ok(lib.hn_graph_create_csr(nv, 2, off, (c_int32 * 2)(1, 0), 1, 0.0, None, byref(h)))
used, total = fake.fake_used(), c_uint64()
for count in lib.hn_tc2_stored, lib.hn_tc_count:
    count.argtypes = [c_void_p, c_void_p, c_void_p, c_void_p]
    ok(count(h, byref(total), None, None))
scratch = fake.fake_used() - used
assert 0 < scratch < 1.25 * 1.125 * (40 * nv + (4 << 20)), scratch / nv
""")


def test_headers_allocate_what_the_library_keeps(fake, tmp_path):
    """The C++ headers' own allocations, on a device filled by a destroyed graph."""
    (tmp_path / "main.cpp").write_text(r"""
#include "hornet/operators.hpp"
extern "C" void fake_device_total(long);
extern "C" long fake_used();
static void keep() {   // the device is full of it
    hn_graph* g = nullptr;
    int64_t off[1001] = {};
    fake_device_total(0);
    (void)hn_memory_trim();
    if (hn_graph_create_csr(1000, 0, off, nullptr, 0, 0.0, nullptr, &g) != HN_OK) throw 1;
    (void)hn_graph_destroy(g);
    fake_device_total(fake_used());
}
int main() {
    keep();
    hornet::COO<> coo(1000);
    keep();
    hornet::CSR<> csr(100, 1000);
    keep();
    int* p = nullptr;
    hornets_nest::gpu::allocate(p, 1000);
    return 0;
}
""")
    lib = os.path.join(ROOT, "hornet_amd")
    exe = str(tmp_path / "main")
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "-O1", "-std=c++17", f"-I{ROOT}/include",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", str(tmp_path / "main.cpp"), "-x", "none",
                    fake, f"{lib}/libhornet_hip.so", "-o", exe, f"-Wl,-rpath,{lib}", f"-Wl,-rpath,{os.path.dirname(fake)}"],
                   check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_package_allocates_what_the_library_keeps(monkeypatch):
    import torch

    import hornet_amd.graph as G
    calls = []

    def empty(n, dtype, device):
        calls.append(n)
        if len(calls) == 1:
            raise torch.OutOfMemoryError("no memory")
        return torch.zeros(n, dtype=dtype)

    monkeypatch.setattr(G, "_dev", lambda: "cpu")
    monkeypatch.setattr(G, "call", lambda name, *a: calls.append(name))
    monkeypatch.setattr(G.torch, "empty", empty)
    assert G._empty(7).shape == (7,) and calls == [7, "hn_memory_trim", 7]
