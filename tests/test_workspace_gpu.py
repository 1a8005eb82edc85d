"""Calls that must not share transient memory: a captured graph and a later, larger call; two streams;
two threads on one stream."""
import threading

import pytest
import torch

from gpu_util import DEV, announce
from nemotron_infer_amd import _lib, ops, synth

pytestmark = pytest.mark.gpu

HIDDEN, INTER = 3136, 12544


def _mlp_weights():
    up, dn = synth.make_weight(INTER, HIDDEN, 41, DEV), synth.make_weight(HIDDEN, INTER, 42, DEV)
    return (torch.ones(HIDDEN, device=DEV), *up, *dn)


def _same(a, b):
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("M", [1, 40, 520])
def test_a_graph_outlives_a_larger_call(M):
    """An eager call and a captured one, then an eager call that needs more transient memory, then
    tensors that take whatever memory was given back: a replay gives the eager bytes and leaves
    those tensors alone."""
    announce("graph_then_larger_call", M)
    w = _mlp_weights()
    x = synth.make_act(M, HIDDEN, 43 + M, DEV)
    want = ops.mlp_forward_fp8(x, *w)
    out = torch.empty_like(x)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=torch.cuda.Stream()):
        ops.mlp_forward_fp8(x, *w, out=out)
    need = _lib.lib().nmi_mlp_workspace_bytes
    assert need(1536, HIDDEN, INTER) > max(need(M, HIDDEN, INTER), 1 << 20)
    ops.mlp_forward_fp8(synth.make_act(1536, HIDDEN, 44, DEV), *w)
    torch.cuda.synchronize()
    fill = [torch.full((max(need(M, HIDDEN, INTER), 1 << 20),), 77, dtype=torch.uint8, device=DEV) for _ in range(4)]
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert _same(out, want)
        assert all(torch.all(t == 77) for t in fill), "the replay wrote into another tensor"
        ops.mlp_forward_fp8(x, *w)                            # eager work between replays


def test_two_streams_and_two_threads():
    """K-split linears (300 x 3136 x 12544: partials, then their sum) and MLP blocks of 40 rows, issued
    on two streams at once and by two threads on one stream: every result is the lone call's."""
    announce("two_streams")
    w = _mlp_weights()
    xs = [synth.make_act(300, INTER, 50 + i, DEV) for i in range(2)]
    ms = [synth.make_act(40, HIDDEN, 60 + i, DEV) for i in range(2)]
    assert _lib.lib().nmi_linear_workspace_bytes(300, HIDDEN, INTER) > 0

    def calls(i, n):
        return [(ops.linear_fp8_w8a16(xs[i], w[3], w[4]), ops.mlp_forward_fp8(ms[i], *w)) for _ in range(n)]

    want = [calls(i, 1)[0] for i in range(2)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    got = [[], []]
    for _ in range(20):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[i] += calls(i, 1)
    torch.cuda.synchronize()
    threads = [threading.Thread(target=lambda i=i: got[i].extend(calls(i, 20))) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i in range(2):
        assert len(got[i]) == 40
        assert all(_same(a, want[i][0]) and _same(b, want[i][1]) for a, b in got[i]), i
