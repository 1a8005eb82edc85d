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


# The four blocks without a workspace, at sizes whose K-split region is more than half of the whole.
BLOCKS = """
W = 1 << 38                                      # a 256-byte aligned address, never touched
ST = 1 << 12                                     # a stream
def mlp(ws, n):
    return L.nmi_mlp_forward_fp8(W, W, W, W, W, W, W, 1536, 3136, 12544, 1e-5, ws, n, ST)
def attn(ws, n):
    return L.nmi_attn_forward_fp8(W, W, W, W, W, W, W, W, W, W, W, 520, W, W, 520, 3136, 40, 8, 1e-5, ws, n, ST)
def mamba_forward(ws, n):
    return L.nmi_mamba_forward_fp8(*[W] * 13, 1, 520, W, W, 3136, 96, 80, 8, 128, 4, 1e-5, ws, n, ST)
def mamba_decode(ws, n):
    return L.nmi_mamba_decode_fp8(*[W] * 15, 24, 3136, 96, 80, 8, 128, 4, 1e-5, ws, n, ST)
full = {"mlp": L.nmi_mlp_workspace_bytes(1536, 3136, 12544), "attn": L.nmi_attn_forward_workspace_bytes(520, 3136, 40, 8),
        "mamba_forward": L.nmi_mamba_forward_workspace_bytes(1, 520, 3136, 96, 80, 8, 128),
        "mamba_decode": L.nmi_mamba_decode_workspace_bytes(24, 3136, 96, 80, 8, 128)}[BLOCK]
call = globals()[BLOCK]
lo, hi = 1, full                                 # the least a caller's workspace may be
while lo < hi:
    mid = (lo + hi) // 2
    lo, hi = (lo, mid) if call(W, mid) == 0 else (mid + 1, hi)
least = lo
hip.stub_take_log()
def kernels():
    return [l[0] for l in launches()]
assert call(W, least) == 0
unsplit = kernels()
assert call(W, full) == 0
split = kernels()
"""


@pytest.mark.parametrize("block", ["mlp", "attn", "mamba_forward", "mamba_decode"])
def test_blocks_without_a_workspace_fall_back_to_the_unsplit_form(host, block):
    """The K split's partials are no reason to fail: where the allocator cannot give the whole
    workspace -- the device is out of memory, or the stream is being captured and no slab has the
    room, when asking for one would end the capture -- the block runs with the smaller one."""
    r = host(f"BLOCK = {block!r}" + BLOCKS + """
slab = lambda n: max(64 * MB, (n + 127) // 128 * 128)
result = {"full": full, "least": least, "split": split, "unsplit": unsplit}
def without(setup):
    L.nmi_alloc_reset()
    setup()
    rc, before = call(None, 0), hip.stub_mallocs()
    k = kernels()
    hip.stub_capturing(0)
    hip.stub_malloc_limit(1 << 60)
    return [rc, k]
result["room"] = without(lambda: None)
# a little less than the whole, of a slab that already holds something
taken = max(0, 64 * MB - full + 4096) if full < 64 * MB else 0
def fill():
    if taken:
        alloc(taken)
def small_device():
    fill()
    hip.stub_malloc_limit(max(least, full - 4096) if not taken else 0)
def capture():
    if taken:
        fill()
    else:
        alloc(least)
        L.nmi_alloc_rewind()
    hip.stub_capturing(1)
result["small_device"] = without(small_device)
result["capture"] = without(capture)
""")
    assert r["least"] < r["full"] and r["unsplit"] != r["split"]
    assert r["room"] == [0, r["split"]]
    assert r["small_device"] == [0, r["unsplit"]], r["small_device"]
    assert r["capture"] == [0, r["unsplit"]], r["capture"]


# Which kernel takes one matrix of N x K below 512 rows (y with row stride N + pad): at the crossings of
# the two models, and where the DMA-fed kernel's tiles end in a ragged band or y's rows are not
# 16-byte aligned.
@pytest.mark.parametrize("M,N,K,pad,kernel", [
    (64, 12544, 3136, 0, "short"), (300, 12544, 3136, 0, "dma"), (200, 3136, 12544, 0, "short"),
    (511, 3136, 12544, 0, "dma"), (511, 3137, 12544, 0, "dma"), (128, 17504, 3136, 0, "short"),
    (129, 17504, 3136, 0, "dma"), (511, 255, 3136, 0, "short"), (511, 256, 3136, 0, "dma"),
    (300, 300, 2048, 0, "short"), (511, 257, 3136, 0, "short"), (511, 384, 3136, 0, "short"),
    (511, 900, 3136, 0, "short"), (511, 1000, 3136, 0, "short"), (511, 1600, 3136, 0, "dma"),
    (200, 9001, 3136, 0, "short"), (511, 9001, 2048, 0, "dma"), (511, 1536, 3136, 0, "dma"),
    (511, 1536, 3136, 3, "short"), (511, 1536, 3136, 8, "dma"),
])
def test_kernel_below_512_rows(host, M, N, K, pad, kernel):
    got = host(f"""
M, N, K, ldy = {M}, {N}, {K}, {N + pad}
W = 1 << 38
n = L.nmi_linear_workspace_bytes(M, N, K)
assert L.nmi_linear_fp8_w8a16_ws(W, K, W, K, W, W, ldy, M, N, K, W if n else None, n, 1 << 12) == 0
result = [l[0] for l in launches()]
""")
    assert ("gemm_short_kernel" if kernel == "short" else "gemm_fp8_w8a16_dma_kernel") in got[0], got


def test_both_kernels_take_some_of_the_gpu_parity_cases(host):
    """tests/test_gemm_split_gpu.py runs these sizes against the oracle as cases on both sides of the
    choice, and the grouped ones as every form of the short-prompt kernel's tiles."""
    one, many, forms = host("""
W, ST = 1 << 38, 1 << 12
def grouped(Ns, M, K):
    arr = (_lib.LinearGroup * len(Ns))(*[_lib.LinearGroup(W, K, W, W, N, N) for N in Ns])
    n = L.nmi_linear_workspace_bytes(M, sum(Ns), K)
    assert L.nmi_linear_fp8_w8a16_grouped(W, K, M, K, arr, len(Ns), W if n else None, n, ST) == 0
    return launches()[0][0]
Ms = (17, 64, 65, 130, 300, 511)
result = [[grouped(Ns, M, K) for Ns, K in (((17500,), 320), ((300,), 5120)) for M in Ms],
          [grouped((1000, 260, 130), M, 1024) for M in Ms],
          [grouped((130, 77, 1, 260), M, K) for M in (17, 32, 33, 64, 65, 128, 129) for K in (64, 1088)]
          + [grouped((30001, 12544, 77, 6800), M, K) for M in (17, 32) for K in (128, 320)]]
""")
    for names in (one, many):
        assert any("gemm_short_kernel" in k for k in names) and any("gemm_fp8_w8a16_dma_kernel" in k for k in names), names
    assert len({k for k in forms if "gemm_short_kernel" in k and "Lb1E" in k}) == 4, set(forms)


def test_linear_workspace_is_enough(host):
    """The bytes the library asks for give the launches that unlimited ones do: one matrix, and up to
    64 rows matrices sharing x, at and between the row tiles of the kernels."""
    bad, asked = host("""
import random
rng = random.Random(5)
W, ST, HUGE = 1 << 38, 1 << 12, 1 << 33
bad, asked = [], {}
def linear(Ns, M, K, n):
    arr = (_lib.LinearGroup * len(Ns))(*[_lib.LinearGroup(W, K, W, W, N, N) for N in Ns])
    assert L.nmi_linear_fp8_w8a16_grouped(W, K, M, K, arr, len(Ns), W, n, ST) == 0
    return launches()
for M in (17, 31, 32, 33, 64, 65, 100, 128, 129, 256, 300, 511):
    for i in range(60):
        K = 64 * rng.choice((1, 5, 16, 32, 49, 80, 120, 196))
        Ns = [rng.choice((1, 130, 300, 1024, 2048, 3136, 5120, 12544, 17504, rng.randint(1, 50000)))]
        if M <= 64 and i % 3 == 0:
            Ns += [rng.randint(1, 9000) for _ in range(rng.randint(1, 3))]
        n = L.nmi_linear_workspace_bytes(M, sum(Ns), K)
        if linear(Ns, M, K, n) != linear(Ns, M, K, HUGE):
            bad.append((M, Ns, K, n))
        asked[M] = max(asked.get(M, 0), n)
result = [bad, asked]
""")
    assert not bad, bad[:5]
    # the short-prompt kernel's one round of 128-row tiles, or one 256 x 256 tile per CU
    assert all(n <= 65536 + (64 << 20) for m, n in asked.items() if int(m) > 64), asked
