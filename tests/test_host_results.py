"""The host side of the synchronous entry points without a GPU: what they
allocate, through a stand-in for the HIP runtime (hip_stub.c) that a child
process loads before the C ABI library.  Kernels do nothing there."""
import os
import subprocess
import sys

import pytest

from dcell_amd import _lib as L

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes as C, sys, threading
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
lib = C.CDLL(sys.argv[2])
lib.dcl_last_error.restype = C.c_char_p
class I3(C.Structure): _fields_ = [("x", C.c_int32), ("y", C.c_int32), ("z", C.c_int32)]
class D3(C.Structure): _fields_ = [("x", C.c_double), ("y", C.c_double), ("z", C.c_double)]
class Win(C.Structure): _fields_ = [("p", I3), ("n", I3), ("d", D3)]
win = Win(I3(0, 0, 0), I3(20, 20, 20), D3(1, 1, 1))
phi, out, count = (C.c_double * 8000)(), (C.c_int32 * 300)(), C.c_int64()
def get(name): return C.c_int.in_dll(stub, name).value
def put(name, v): C.c_int.in_dll(stub, name).value = v
def band(static=False, count=count):
    f = lib.dcl_band_compact_static if static else lib.dcl_band_compact
    return f(C.byref(phi), C.byref(win), C.c_double(1.0), 0, C.byref(out), C.c_int64(100), C.byref(count), None)
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    d = tmp_path_factory.mktemp("hip_stub")
    so, ver = str(d / "libamdhip64.so.7"), d / "stub.map"
    ver.write_text("hip_4.2 { global: *; };\nhip_4.3 { global: hipGraph*; } hip_4.2;\n")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-std=gnu11", "-Wl,-soname,libamdhip64.so.7",
                    f"-Wl,--version-script={ver}", "-o", so, os.path.join(HERE, "hip_stub.c"), "-lpthread"],
                   check=True)
    return so


def run(stub, code):
    r = subprocess.run([sys.executable, "-c", PRELUDE + code, stub, L.LIB_PATH], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


def test_static_band_compaction_allocates_nothing(stub):
    """As the first call of a process, when a launch fails, and with many calls
    under way at once."""
    run(stub, """
assert band(static=True) == 0, lib.dcl_last_error()
assert get("stub_launches") == 4
put("stub_fail_launch", 1)
assert band(static=True) != 0
put("stub_fail_launch", 0)
stub.stub_reset_hold(80)
ts = [threading.Thread(target=lambda: band(static=True, count=C.c_int64())) for _ in range(80)]
[t.start() for t in ts]
[t.join() for t in ts]
assert get("stub_allocs") == get("stub_frees") == 0, (get("stub_allocs"), get("stub_frees"))
""")


def test_result_words_come_back(stub):
    """The 64 pinned words are one allocation; a call that fails between taking
    its word and waiting for the stream gives it back; with all of them taken a
    call allocates its own and frees it; a word whose stream cannot be waited
    for stays taken."""
    run(stub, """
assert band() == 0, lib.dcl_last_error()
assert get("stub_host_allocs") == 1
put("stub_fail_launch", 1)
for _ in range(200):
    assert band() != 0
put("stub_fail_launch", 0)
assert band() == 0 and get("stub_host_allocs") == 1
# 70 calls under way at once: none returns before the last waits for its stream
stub.stub_reset_hold(70)
rc = []
ts = [threading.Thread(target=lambda: rc.append(band(count=C.c_int64()))) for _ in range(70)]
[t.start() for t in ts]
[t.join() for t in ts]
stub.stub_reset_hold(0)
assert rc == [0] * 70
assert get("stub_host_allocs") == 1 + 6 and get("stub_host_frees") == 6
assert band() == 0 and get("stub_host_allocs") == 7
put("stub_fail_sync", 1)
for _ in range(64):
    assert band() != 0
assert get("stub_host_allocs") == 7
put("stub_fail_sync", 0)
assert band() == 0
assert get("stub_host_allocs") == 8 and get("stub_host_frees") == 7
""")
