"""The DMA-fed GEMM's tile rows (128, 192, 256) and its K split (float32 partial tiles in the
workspace, added by a second kernel) against the oracle, at the edges of the tiles."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from gpu_util import DEV, announce, assert_parity, bits, oracle_bits, s_to_dev, w_to_dev, x_to_dev
from nemotron_infer_amd import _lib, ops, synth

pytestmark = pytest.mark.gpu

KNOBS = ("gemm.bm", "gemm.splits", "gemm.tile", "gemm.sk")


@pytest.fixture(autouse=True)
def _reset():
    yield
    for k in KNOBS:
        _lib.tuning_set(k, 0)


def _case(M, N, K, seed, scales="log_uniform"):
    w, s = synth.make_weight(N, K, seed, "cpu", scales=scales)
    x = synth.make_act(M, K, seed + 1, "cpu")
    return x.view(torch.int16).numpy().view(np.uint16), w.numpy(), s.numpy()


def _call(xd, wd, sd, y, ldy, M, N, K, ws, nbytes):
    _lib.check(_lib.lib().nmi_gemm_fp8_w8a16(xd.data_ptr(), K, wd.data_ptr(), K, sd.data_ptr(), y.data_ptr(), ldy, M,
                                             N, K, None if ws is None else ws.data_ptr(), nbytes,
                                             torch.cuda.current_stream().cuda_stream), "gemm")


# M around the tile rows and the 32-row strips of the second kernel, ragged N (one and two column
# bands), one k tile per split and uneven splits.
@pytest.mark.parametrize("M,N,K", [(512, 256, 320), (513, 300, 640), (576, 257, 704), (767, 40, 320), (1, 264, 320),
                                   (97, 513, 1024)])
@pytest.mark.parametrize("bm", [128, 192, 256])
def test_tile_rows_and_splits(bm, M, N, K):
    x, w, s = _case(M, N, K, bm + M + N + K)
    xd, wd, sd = x_to_dev(x), w_to_dev(w), s_to_dev(s)
    ref = oracle_bits(x, w, s)
    L = _lib.lib()
    _lib.tuning_set("gemm.tile", 24)
    _lib.tuning_set("gemm.bm", bm)
    _lib.tuning_set("gemm.sk", 2)                  # not the stream-K form, whose flags must be zero
    unsplit = None
    for sp in (1, 2, 5):
        _lib.tuning_set("gemm.splits", sp)
        need = L.nmi_linear_workspace_bytes(max(M, 512), N, K)
        announce("gemm_split", bm, M, N, K, sp, need)
        ws = torch.full((max(need, 256),), 255, dtype=torch.uint8, device=DEV)   # NaN where not written
        ys = []
        # contiguous y, y with an odd row stride and 2-byte offset, and a workspace of the
        # flag region only
        for ldy, off, nbytes in ((N, 0, need), (N + 3, 1, need), (N, 0, min(need, 65536))):
            buf = torch.full((M, ldy), 5.0, dtype=torch.bfloat16, device=DEV)
            _call(xd, wd, sd, buf[:, off:], ldy, M, N, K, ws, nbytes)
            torch.cuda.synchronize()
            ys.append(bits(buf[:, off:off + N]))
            assert torch.all(buf[:, :off] == 5.0) and torch.all(buf[:, off + N:] == 5.0)
        assert torch.all(ws[:min(need, 65536)] == 255), "flag region written"
        assert_parity(ys[0], ref, f"bm={bm} splits={sp}", per_row_scales=True)
        assert np.array_equal(ys[0], ys[1])
        unsplit = ys[0] if unsplit is None else unsplit
        assert np.array_equal(ys[2], unsplit), "without room for the partials: the unsplit sums"


def test_automatic_split_in_the_mlp_block_and_a_graph():
    """M = 520 at the model's sizes: down_proj (K = 12544) is split.  relu^2, the residual (in place
    too) and graph replays give the composition's bytes; a workspace without room for the
    partials is accepted and stays within the parity of another summation order."""
    M, hidden, inter = 520, 3136, 12544
    announce("gemm_split_mlp", M, hidden, inter)
    L = _lib.lib()
    assert L.nmi_linear_workspace_bytes(M, hidden, inter) > 65536
    assert L.nmi_linear_workspace_needs_zero(M) == 0 and L.nmi_linear_workspace_needs_zero(511) == 1
    up, ups = synth.make_weight(inter, hidden, 31, DEV)
    dn, dns = synth.make_weight(hidden, inter, 32, DEV)
    nw = torch.ones(hidden, device=DEV)
    x = synth.make_act(M, hidden, 33, DEV)
    h = ops.rmsnorm_bf16(x, nw)
    u = ops.linear_fp8_w8a16(h, up, ups)
    r = torch.relu(u)
    want = x + ops.linear_fp8_w8a16(r * r, dn, dns)
    got = ops.mlp_forward_fp8(x, nw, up, ups, dn, dns)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    xi = x.clone()
    ops.mlp_forward_fp8(xi, nw, up, ups, dn, dns, out=xi)
    assert torch.equal(xi.view(torch.int16), want.view(torch.int16)), "in place"
    out = torch.empty_like(x)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        ops.mlp_forward_fp8(x, nw, up, ups, dn, dns, out=out)
        lin = ops.linear_fp8_w8a16(r * r, dn, dns)
    for _ in range(3):
        out.zero_()
        lin.zero_()
        ops.mlp_forward_fp8(x, nw, up, ups, dn, dns)          # eager work between replays
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), want.view(torch.int16))
        assert torch.equal((x + lin).view(torch.int16), want.view(torch.int16))
    need = L.nmi_mlp_workspace_bytes(M, hidden, inter)
    least = need - (L.nmi_linear_workspace_bytes(M, hidden, inter) + 255) // 256 * 256
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    for nbytes, ok in ((need - 1, True), (least, True), (least - 1, False)):
        rc = L.nmi_mlp_forward_fp8(x.data_ptr(), nw.data_ptr(), up.data_ptr(), ups.data_ptr(), dn.data_ptr(),
                                   dns.data_ptr(), out.data_ptr(), M, hidden, inter, 1e-5, ws.data_ptr(), nbytes, None)
        assert (rc == _lib.NMI_OK) == ok, (nbytes, rc)
        torch.cuda.synchronize()
        if ok:
            d = (out.double() - want.double()).norm() / want.double().norm()
            assert d < 2e-3, d                               # rounding flips of another float32 order


# The choice between the short-prompt and the DMA-fed kernel at M < 512 (one matrix, and matrices
# sharing x), on both sides of it: with a workspace, without one, and with one too small.  (Which
# kernel takes which of these: test_host_runtime_cpu.py.)
@pytest.mark.parametrize("M", [17, 64, 65, 130, 300, 511])
@pytest.mark.parametrize("Ns,K", [((17500,), 320), ((1000, 260, 130), 1024), ((300,), 5120)])
def test_below_512_rows(M, Ns, K):
    announce("gemm_below_512", M, Ns, K)
    cases = [_case(M, N, K, 13 * i + M + N + K) for i, N in enumerate(Ns)]
    x = cases[0][0]
    xd = x_to_dev(x)
    wd = [(w_to_dev(w), s_to_dev(s)) for _, w, s in cases]
    L = _lib.lib()
    need = L.nmi_linear_workspace_bytes(M, sum(Ns), K)
    ws = torch.full((max(need, 256),), 255, dtype=torch.uint8, device=DEV)
    refs = [oracle_bits(x, w, s) for _, w, s in cases]
    arr = (_lib.LinearGroup * len(Ns))()
    for nbytes in (need, min(need, 65536), 0):
        ys = [torch.full((M, N), 5.0, dtype=torch.bfloat16, device=DEV) for N in Ns]
        for i, ((w, s), y) in enumerate(zip(wd, ys)):
            arr[i] = _lib.LinearGroup(w.data_ptr(), w.stride(0), s.data_ptr(), y.data_ptr(), y.stride(0), w.shape[0])
        _lib.check(L.nmi_linear_fp8_w8a16_grouped(xd.data_ptr(), K, M, K, arr, len(Ns),
                                                  ws.data_ptr() if nbytes else None, nbytes, None), "grouped")
        torch.cuda.synchronize()
        assert torch.all(ws[:min(need, 65536)] == 255), "flag region written"
        for i, (y, ref) in enumerate(zip(ys, refs)):
            assert_parity(bits(y), ref, f"M={M} group {i} ws={nbytes}", per_row_scales=True)


# Matrices sharing x below 512 rows as one launch: every row-tile form of the short-prompt kernel but
# the widest (the next test), row counts that are no multiple of 4 (the partials after them are unaligned), one k tile (no split), many.
@pytest.mark.parametrize("M", [17, 32, 33, 64, 65, 128, 129])
@pytest.mark.parametrize("K", [64, 1088])
def test_grouped_short(M, K):
    Ns = (130, 77, 1, 260)
    announce("gemm_grouped_short", M, Ns, K)
    cases = [_case(M, N, K, 19 * i + M + N + K) for i, N in enumerate(Ns)]
    xd = x_to_dev(cases[0][0])
    wd = [(w_to_dev(w), s_to_dev(s)) for _, w, s in cases]
    L = _lib.lib()
    total = sum(Ns)
    need = L.nmi_linear_workspace_bytes(M, total, K)
    ws = torch.full((max(need, 256),), 255, dtype=torch.uint8, device=DEV)
    ybig = torch.full((M, total + 3), 5.0, dtype=torch.bfloat16, device=DEV)
    offs = np.cumsum((0,) + Ns)
    arr = (_lib.LinearGroup * len(Ns))()
    for i, (w, s) in enumerate(wd):
        y = ybig[:, offs[i]:offs[i + 1]]
        arr[i] = _lib.LinearGroup(w.data_ptr(), w.stride(0), s.data_ptr(), y.data_ptr(), y.stride(0), w.shape[0])
    _lib.check(L.nmi_linear_fp8_w8a16_grouped(xd.data_ptr(), K, M, K, arr, len(Ns), ws.data_ptr(), need, None), "grouped")
    torch.cuda.synchronize()
    for i, (_, w, s) in enumerate(cases):
        assert_parity(bits(ybig[:, offs[i]:offs[i + 1]]), oracle_bits(cases[0][0], w, s), f"M={M} K={K} group {i}",
                      per_row_scales=True)
    assert torch.all(ybig[:, total:] == 5.0)
    assert torch.all(ws[:min(need, 65536)] == 255), "flag region written"


# The 256 x 32 tiles, which only few rows of x against some 49000 weight rows and more take: ragged
# matrices, a matrix within one tile, two and five k tiles (too few to split).
@pytest.mark.parametrize("M", [17, 32])
@pytest.mark.parametrize("K", [128, 320])
def test_grouped_short_wide_tiles(M, K):
    Ns = (30001, 12544, 77, 6800)
    announce("gemm_grouped_short_wide", M, Ns, K)
    cases = [_case(M, N, K, 23 * i + M + K) for i, N in enumerate(Ns)]
    xd = x_to_dev(cases[0][0])
    wd = [(w_to_dev(w), s_to_dev(s)) for _, w, s in cases]
    ys = [torch.full((M, N + 3), 5.0, dtype=torch.bfloat16, device=DEV) for N in Ns]
    arr = (_lib.LinearGroup * len(Ns))(*[_lib.LinearGroup(w.data_ptr(), K, s.data_ptr(), y.data_ptr(), y.stride(0), N)
                                         for (w, s), y, N in zip(wd, ys, Ns)])
    _lib.check(_lib.lib().nmi_linear_fp8_w8a16_grouped(xd.data_ptr(), K, M, K, arr, len(Ns), None, 0, None), "grouped")
    torch.cuda.synchronize()
    for i, ((_, w, s), y) in enumerate(zip(cases, ys)):
        assert_parity(bits(y[:, :-3]), oracle_bits(cases[0][0], w, s), f"M={M} K={K} group {i}", per_row_scales=True)
        assert torch.all(y[:, -3:] == 5.0)


# Groups of ragged column bands with K split in every tile height.
@pytest.mark.parametrize("bm", [128, 192, 256])
def test_grouped_split_tile_rows(bm):
    M, Ns, K = 200, (300, 40, 257), 640
    announce("gemm_grouped_split", bm, M, Ns, K)
    cases = [_case(M, N, K, 17 * i + bm + N) for i, N in enumerate(Ns)]
    xd = x_to_dev(cases[0][0])
    wd = [(w_to_dev(w), s_to_dev(s)) for _, w, s in cases]
    refs = [oracle_bits(cases[0][0], w, s) for _, w, s in cases]
    _lib.tuning_set("gemm.sk", 2)
    _lib.tuning_set("gemm.bm", bm)
    _lib.tuning_set("gemm.splits", 3)
    L = _lib.lib()
    total = sum(Ns)
    need = L.nmi_linear_workspace_bytes(M, total, K)
    assert need > 0
    ws = torch.full((need,), 255, dtype=torch.uint8, device=DEV)
    ybig = torch.full((M, total + 3), 5.0, dtype=torch.bfloat16, device=DEV)
    offs = np.cumsum((0,) + Ns)
    arr = (_lib.LinearGroup * len(Ns))()
    for i, (w, s) in enumerate(wd):
        y = ybig[:, offs[i]:offs[i + 1]]
        arr[i] = _lib.LinearGroup(w.data_ptr(), w.stride(0), s.data_ptr(), y.data_ptr(), y.stride(0), w.shape[0])
    for split in (3, 0):
        _lib.tuning_set("gemm.splits", split)
        ybig[:, :total] = 5.0
        _lib.check(L.nmi_linear_fp8_w8a16_grouped(xd.data_ptr(), K, M, K, arr, len(Ns), ws.data_ptr(), need, None), "g")
        torch.cuda.synchronize()
        for i, ref in enumerate(refs):
            assert_parity(bits(ybig[:, offs[i]:offs[i + 1]]), ref, f"bm={bm} group {i}", per_row_scales=True)
        assert torch.all(ybig[:, total:] == 5.0)


@pytest.mark.parametrize("batch", [16, 17, 33])
def test_mamba_decode_batch_workspace(batch):
    """The Mamba-2 decode block where its projections turn into GEMMs (batch 17): with the whole
    workspace and without the part for the K split (the older size) it stays within the flips of
    another float32 order of the composition of the library's calls; states the same bytes."""
    H, P, G, hidden = 96, 80, 8, 3136
    inter, conv_dim = H * P, H * P + 2 * G * 128
    announce("mamba_decode_batch_ws", batch)
    g = torch.Generator(device=DEV).manual_seed(50 + batch)
    f = {"device": DEV, "generator": g}
    iw, isc = synth.make_weight(inter + conv_dim + H, hidden, 61, DEV)
    ow, osc = synth.make_weight(hidden, inter, 62, DEV)
    prm = [0.3 * torch.randn((conv_dim, 4), **f), 0.1 * torch.randn(conv_dim, **f), torch.rand(H, **f),
           torch.randn(H, **f), 0.5 * torch.randn(H, **f), 1.0 + 0.1 * torch.randn(inter, **f)]
    nw = torch.ones(hidden, device=DEV)
    x = synth.make_act(batch, hidden, 63, DEV)
    cs = torch.randn((batch, conv_dim, 3), **f)
    ss = 0.1 * torch.randn((batch, H, P, 128), **f)
    h = ops.rmsnorm_bf16(x, nw)
    c0, s0 = cs.clone(), ss.clone()
    proj = ops.linear_fp8_w8a16(h, iw, isc)
    _, gg = ops.mamba_mixer_decode(proj, *prm, c0, s0, H, P, G)
    want = x + ops.linear_fp8_w8a16(gg, ow, osc)
    L = _lib.lib()
    need = L.nmi_mamba_decode_workspace_bytes(batch, hidden, H, P, G, 128)
    r256 = lambda b: (b + 255) // 256 * 256  # noqa: E731
    least = r256(batch * 17504 * 2) + 2 * r256(batch * inter * 2) + r256(batch * hidden * 2)
    assert need >= least and (need > least) == (batch > 16)
    ws = torch.full((need,), 255, dtype=torch.uint8, device=DEV)
    for nbytes in (need, least, least - 1):
        c1, s1, out = cs.clone(), ss.clone(), torch.empty_like(x)
        rc = L.nmi_mamba_decode_fp8(x.data_ptr(), nw.data_ptr(), iw.data_ptr(), isc.data_ptr(),
                                    *[t.data_ptr() for t in prm], ow.data_ptr(), osc.data_ptr(), c1.data_ptr(),
                                    s1.data_ptr(), out.data_ptr(), batch, hidden, H, P, G, 128, 4, 1e-5, ws.data_ptr(),
                                    nbytes, None)
        assert (rc == _lib.NMI_OK) == (nbytes >= least), (nbytes, rc)
        torch.cuda.synchronize()
        if nbytes == need:
            assert torch.equal(out.view(torch.int16), want.view(torch.int16))
            assert torch.equal(c1, c0) and torch.equal(s1, s0)
        elif nbytes == least:
            # a few flipped roundings (2^-9 relative each) among the block's values
            assert (out.double() - want.double()).norm() / want.double().norm() < 2e-3
            assert (s1 - s0).norm() / s0.norm() < 1e-3
