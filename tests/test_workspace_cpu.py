"""Where the torch front end's transient device memory comes from (nemotron_infer_amd/ops.py), no GPU
needed: each call takes its own from torch's allocator and keeps none of it.  Memory kept between
calls would be shared by every stream and thread, and a HIP graph captured with it would go on
writing into it after a larger call had replaced it.  The library is replaced by a recorder."""
import ctypes
import weakref

import pytest
import torch

from nemotron_infer_amd import _lib, ops

NEED = 1_200_000
FLAGS = _lib.NMI_WS_ERROR_OFFSET + 4


class Recorder:
    """Stands in for libnmi.so: every workspace is NEED bytes; launches note their arguments and the
    first bytes of the workspace they were given."""

    def __init__(self, needs_zero=0):
        self.needs_zero, self.launches = needs_zero, []

    def __getattr__(self, name):
        if name.endswith("workspace_bytes"):
            return lambda *a: NEED
        if name == "nmi_linear_workspace_needs_zero":
            return lambda M: self.needs_zero

        def launch(*args):
            at = next(i for i in range(len(args) - 1) if args[i + 1] == NEED)
            self.launches.append((name, args[at], ctypes.string_at(args[at], FLAGS + 16)))
            return _lib.NMI_OK
        return launch


@pytest.fixture
def made(monkeypatch):
    """The uint8 tensors torch.empty makes (weak), filled with 255."""
    refs, empty = [], torch.empty

    def spy(*a, **kw):
        t = empty(*a, **kw)
        if t.dtype == torch.uint8:
            t.fill_(255)
            refs.append((weakref.ref(t), t.data_ptr()))
        return t
    monkeypatch.setattr(torch, "empty", spy)
    monkeypatch.setattr(ops, "_check_device", lambda *ts: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    return refs


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
def test_workspaces_belong_to_one_call(call, made, monkeypatch):
    lib = Recorder()
    monkeypatch.setattr(_lib, "lib", lambda: lib)
    for n in (1, 2):
        before = len(made)
        out = CALLS[call]()
        assert out is not None and len(lib.launches) == n
        mine = {ptr: ref for ref, ptr in made[before:]}
        assert lib.launches[-1][1] in mine, "not from torch's allocator in this call"
        assert mine[lib.launches[-1][1]]() is None, "kept after the call"


@pytest.mark.parametrize("M,needs_zero,zeroed", [(600, 1, True), (600, 0, False), (24, 1, False)])
def test_only_stream_k_flags_are_cleared(M, needs_zero, zeroed, made, monkeypatch):
    """From M = 512 the flag region starts at zero where the library says so (the stream-K form);
    below, the kernels leave it alone, so it is not cleared on every call."""
    lib = Recorder(needs_zero)
    monkeypatch.setattr(_lib, "lib", lambda: lib)
    ops.linear_fp8_w8a16(_bf(M, 64), *_mat(32, 64))
    head = lib.launches[0][2]
    assert head == (b"\0" * FLAGS if zeroed else b"\xff" * FLAGS) + b"\xff" * 16
