"""Where the torch front end's transient device memory comes from (nemotron_infer_amd/ops.py), no GPU
needed.  Memory shared by streams or threads would be overwritten by the other's call, and a HIP
graph captured with memory that a larger call replaces would go on writing into it: so what is kept
between calls is kept per stream, out of reach while a call has it, and never under capture.  The
library is replaced by a recorder."""
import ctypes
import weakref

import pytest
import torch

from nemotron_infer_amd import _lib, ops

SMALL, LARGE = 1_200_000, ops._KEEP_BYTES + 512
FLAGS = _lib.NMI_WS_ERROR_OFFSET + 4


class Recorder:
    """Stands in for libnmi.so: every workspace is `need` bytes; launches note the workspace they were
    given and its first bytes, and call `during`."""

    def __init__(self, need=SMALL, needs_zero=0):
        self.need, self.needs_zero, self.launches, self.during = need, needs_zero, [], None

    def __getattr__(self, name):
        if name.endswith("workspace_bytes"):
            return lambda *a: self.need
        if name == "nmi_linear_workspace_needs_zero":
            return lambda M: self.needs_zero

        def launch(*args):
            at = next(i for i in range(len(args) - 1) if args[i + 1] == self.need)
            self.launches.append((name, args[at], ctypes.string_at(args[at], FLAGS + 16)))
            during, self.during = self.during, None
            if during:
                during()
            return _lib.NMI_OK
        return launch


@pytest.fixture
def env(monkeypatch):
    """The uint8 tensors torch.empty makes (weak, filled with 255), and the stream and capture state
    that the front end sees."""
    class Env:
        made, stream, capturing, lib = [], 0, False, Recorder()
    e, empty = Env(), torch.empty
    e.made = []

    def spy(*a, **kw):
        t = empty(*a, **kw)
        if t.dtype == torch.uint8:
            t.fill_(255)
            e.made.append((weakref.ref(t), t.data_ptr()))
        return t
    monkeypatch.setattr(torch, "empty", spy)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: e.capturing)
    monkeypatch.setattr(ops, "_check_device", lambda *ts: None)
    monkeypatch.setattr(ops, "_stream", lambda: e.stream)
    monkeypatch.setattr(ops, "_kept", {})
    monkeypatch.setattr(_lib, "lib", lambda: e.lib)
    return e


def _bf(*shape):
    return torch.zeros(shape, dtype=torch.bfloat16)


def _mat(n, k):
    return torch.zeros((n, k), dtype=torch.uint8), torch.ones(n)


HID, H, P, G = 128, 4, 32, 1
CONV = H * P + 2 * G * 128
MAMBA = [torch.zeros((CONV, 4)), torch.zeros(CONV), torch.zeros(H), torch.zeros(H), torch.zeros(H), torch.zeros(H * P)]
ATTN = [t for n, k in ((256, HID), (128, HID), (128, HID), (HID, 256)) for t in _mat(n, k)]
CALLS = {
    "linear_m24": lambda: ops.linear_fp8_w8a16(_bf(24, 64), *_mat(32, 64)),
    "linear_m600": lambda: ops.linear_fp8_w8a16(_bf(600, 64), *_mat(32, 64)),
    "grouped_m24": lambda: ops.linear_fp8_w8a16_grouped(_bf(24, 64), [_mat(32, 64), _mat(16, 64)]),
    "gemm_m24": lambda: ops.gemm_fp8_w8a16(_bf(24, 64), *_mat(32, 64)),
    "mlp": lambda: ops.mlp_forward_fp8(_bf(24, HID), torch.ones(HID), *_mat(256, HID), *_mat(HID, 256)),
    "sdpa_decode": lambda: ops.sdpa_decode_bf16(_bf(2, 128), _bf(1, 9, 128), _bf(1, 9, 128), _bf(1, 128), _bf(1, 128), 5),
    "attn_decode": lambda: ops.attn_decode_fp8(_bf(1, HID), torch.ones(HID), *ATTN, _bf(1, 9, 128), _bf(1, 9, 128), 5),
    "attn_forward": lambda: ops.attn_forward_fp8(_bf(24, HID), torch.ones(HID), *ATTN),
    "mamba_decode": lambda: ops.mamba_decode_fp8(_bf(2, HID), torch.ones(HID), *_mat(H * P + CONV + H, HID), *MAMBA,
                                                 *_mat(HID, H * P), torch.zeros((2, CONV, 3)),
                                                 torch.zeros((2, H, P, 128)), H, P, G),
    "mamba_forward": lambda: ops.mamba_forward_fp8(_bf(24, HID), torch.ones(HID), *_mat(H * P + CONV + H, HID), *MAMBA,
                                                   *_mat(HID, H * P), H, P, G, batch=2),
}


@pytest.mark.parametrize("call", CALLS)
@pytest.mark.parametrize("need,capturing", [(LARGE, False), (SMALL, True)])
def test_large_and_captured_memory_belongs_to_one_call(call, need, capturing, env):
    env.lib, env.capturing = Recorder(need), capturing
    for n in (1, 2):
        before = len(env.made)
        CALLS[call]()
        assert len(env.lib.launches) == n
        mine = {ptr: ref for ref, ptr in env.made[before:]}
        assert env.lib.launches[-1][1] in mine, "not from torch's allocator in this call"
        assert mine[env.lib.launches[-1][1]]() is None and not ops._kept, "kept after the call"


@pytest.mark.parametrize("call", CALLS)
def test_small_memory_is_kept_for_its_stream_only(call, env):
    """The same memory for the next call on the stream, other memory on another stream, for a call
    that begins while one is under way on the same stream (a second thread), and under capture;
    a larger call replaces what its own stream keeps; every call is told what it asked for."""
    lib = env.lib

    def run(stream=0):
        env.stream = stream
        CALLS[call]()
        return lib.launches[-1][1]

    first = run()
    assert run() == first
    other = run(stream=64)
    assert other != first and run() == first and run(stream=64) == other
    lib.during = run                                  # begins before the outer call's launch returns
    outer = len(lib.launches)
    run()
    assert lib.launches[outer][1] == first and lib.launches[outer + 1][1] != first
    env.capturing = True
    kept = dict(ops._kept)
    assert run() not in [t.data_ptr() for t in kept.values()] and ops._kept == kept
    env.capturing = False
    lib.need = 3 * SMALL
    run()
    assert sorted(ops._kept) == [(None, 0), (None, 64)] and ops._kept[None, 0].numel() == 3 * SMALL
    assert ops._kept[None, 64].data_ptr() == other


def test_kept_memory_is_bounded(env):
    for stream in range(2 * ops._KEEP_STREAMS):
        env.stream = 64 * stream
        for need in (SMALL, LARGE, 2 * SMALL):
            env.lib.need = need
            ops.linear_fp8_w8a16(_bf(24, 64), *_mat(32, 64))
    assert len(ops._kept) == ops._KEEP_STREAMS
    assert all(t.numel() == 2 * SMALL for t in ops._kept.values())


@pytest.mark.parametrize("M,needs_zero,zeroed", [(600, 1, True), (600, 0, False), (24, 1, False)])
def test_only_stream_k_flags_are_cleared(M, needs_zero, zeroed, env):
    """From M = 512 the flag region starts at zero where the library says so (the stream-K form);
    below, the kernels leave it alone, so it is not cleared on every call."""
    env.lib = Recorder(SMALL, needs_zero)
    ops.linear_fp8_w8a16(_bf(M, 64), *_mat(32, 64))
    head = env.lib.launches[0][2]
    assert head == (b"\0" * FLAGS if zeroed else b"\xff" * FLAGS) + b"\xff" * 16
