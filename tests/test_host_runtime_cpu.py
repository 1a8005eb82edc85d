"""Host code of libnmi.so on a stand-in for the HIP runtime (hip_host_stub.cpp), no GPU needed: device
memory it asks for, and the kernels it would launch.  Each case is a process of its own, so that the
library binds to the stand-in."""
import json
import os
import subprocess
import sys

import pytest

from tests.conftest import ROOT

PRELUDE = """
import ctypes, json, sys
hip = ctypes.CDLL({stub!r}, mode=ctypes.RTLD_GLOBAL)
hip.stub_take_log.restype = ctypes.c_char_p
hip.stub_malloc_limit.argtypes = [ctypes.c_size_t]
from nemotron_infer_amd import _lib
L = _lib.lib()
MB = 1 << 20

def launches():
    '''[(kernel, grid x, y, z, threads)] since the last call'''
    return [(l.rsplit(" ", 4)[0], *map(int, l.split()[-4:])) for l in hip.stub_take_log().decode().splitlines()]

def alloc(nbytes):
    p = ctypes.c_void_p()
    rc = L.nmi_alloc(nbytes, ctypes.byref(p))
    return rc, p.value

def slabs():
    n = ctypes.c_size_t()
    L.nmi_alloc_stats(None, ctypes.byref(n))
    return n.value
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    stub = str(tmp_path_factory.mktemp("stub") / "libhipstub.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", "-o", stub,
                    os.path.join(ROOT, "tests", "hip_host_stub.cpp")], check=True, timeout=120)

    def run(body):
        """The value that body (after PRELUDE) leaves in `result`."""
        code = PRELUDE.format(stub=stub) + body + "\nprint(json.dumps(result))\n"
        r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr
        return json.loads(r.stdout.splitlines()[-1])
    return run


def test_bump_allocator_reuses_any_later_slab(host):
    """Two sequences in turn, each after a rewind: one leaves an 80 MB slab behind the first, the
    other asks for 110 MB, which fits neither.  The slab made for it serves all later rounds, and
    the first sequence keeps its own addresses."""
    rounds = host("""
result = []
for _ in range(4):
    row = []
    for seq in ([10 * MB, 80 * MB], [110 * MB]):
        L.nmi_alloc_rewind()
        got = [alloc(n) for n in seq]
        assert all(rc == 0 for rc, _ in got)
        row.append([p for _, p in got])
    result.append([row, slabs(), hip.stub_mallocs()])
""")
    assert rounds[0][1] == 3
    assert all(r == rounds[0] for r in rounds), rounds
