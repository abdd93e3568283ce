"""Ways to the same sums on the bf16 MFMA: the tiles of the bf16 GEMM among each
other (LIGHTX2V_HIP_BF16_CFG), and a Q8 / Q4 / FP8 weight written out as bf16
first against dequantization inside the GEMM (LIGHTX2V_HIP_W16_EXPAND), also
in graphs and without allocations.  All contract the same bf16 values in the
same 16-element steps in the same order, so outputs agree bit for bit."""

import numpy as np
import pytest

import lightx2v_hip as H
import oracle as O
from helpers import W16_TIGHT, assert_close, normal, oracle_w16, u32

pytestmark = pytest.mark.gpu


def _run(be, x, w, b, act, M, N, ydt):
    y = be.alloc((M + 1) * N, ydt)
    be.write(y, np.full((M + 1) * N, np.nan, np.float32))
    be.profile_reset()
    be.profile_enable(True)
    try:
        be.linear(x, 1, M, w, b, act, y, 0)
        names = list(be.profile_stats())
    finally:
        be.profile_enable(False)
        be.profile_reset()
    v = be.download(y).reshape(M + 1, N)
    assert np.isnan(v[M]).all() and not np.isnan(v[:M]).any()
    return v[:M], names


# K of two, three and many stages; one row, tile edges, more tiles than CUs
@pytest.mark.parametrize("M,K,N", [(1, 128, 256), (255, 192, 512), (257, 1536, 256), (2500, 128, 7936), (600, 320, 768)])
@pytest.mark.parametrize("act", [H.ACT_NONE, H.ACT_GELU_TANH])
def test_bf16_persistent_tile_equals_tiles(be, monkeypatch, act, M, K, N):
    monkeypatch.setenv("LIGHTX2V_HIP_ROWS", "0")
    wf, xf, bf = normal(4401 + N, N * K, 0.02), normal(4402, (M + 1) * K), normal(4403, N, 0.01)
    w, x, b = be.weight(wf, N, K), be.alloc((M + 1) * K, H.DTYPE_BF16), be.upload(bf)
    be.write(x, xf)
    out = []
    for cfg in ("0", "5"):
        monkeypatch.setenv("LIGHTX2V_HIP_BF16_CFG", cfg)
        out.append(_run(be, x, w, b if M != 257 else None, act, M, N, H.DTYPE_BF16)[0])
    assert np.array_equal(u32(out[0]), u32(out[1]))
    p = np.unique(np.append(np.arange(0, M, 97), M - 1))
    ref = oracle_w16(O.bf16_round(xf).reshape(M + 1, K)[1:][p], wf.reshape(N, K), bf if M != 257 else None, act)
    assert_close(out[1][p], ref, W16_TIGHT[0] + 2.0**-8, W16_TIGHT[1] + 2.0**-7 * np.abs(ref).max(), what="vs oracle")


# One row and around a 64-row tile, past two; K of one stage, below and past the ring's four slots
@pytest.mark.parametrize("K", [64, 192, 320])
@pytest.mark.parametrize("M,N", [(1, 33), (63, 128), (64, 64), (65, 130), (129, 264), (300, 513)])
def test_bf16_tiles_agree(be, monkeypatch, M, N, K):
    """Every one-shot tile (256 x 128, 128 x 256, 128 x 128, 64 x 128, 64 x 64)
    against the first, bit for bit, and against the oracle."""
    monkeypatch.setenv("LIGHTX2V_HIP_ROWS", "0")
    wf, xf, bf = normal(4451 + N, N * K, 0.02), normal(4452 + M, (M + 1) * K), normal(4453, N, 0.01)
    w, x, b = be.weight(wf, N, K), be.alloc((M + 1) * K, H.DTYPE_BF16), be.upload(bf)
    be.write(x, xf)
    ref = oracle_w16(O.bf16_round(xf).reshape(M + 1, K)[1:], wf.reshape(N, K), bf, 1)
    for ydt in (H.DTYPE_F32, H.DTYPE_BF16):
        out = []
        for cfg in range(5):
            monkeypatch.setenv("LIGHTX2V_HIP_BF16_CFG", str(cfg))
            out.append(_run(be, x, w, b, H.ACT_GELU_TANH, M, N, ydt)[0])
            assert np.array_equal(u32(out[0]), u32(out[-1])), (cfg, ydt)
        if ydt == H.DTYPE_F32:
            assert_close(out[0], ref, *W16_TIGHT, what=f"{M}x{K}->{N}")
        else:
            assert np.array_equal(u32(out[0]), u32(O.bf16_round(f32).reshape(M, N)))
        f32 = out[0]


@pytest.mark.parametrize("M,K,N", [(1, 64, 33), (300, 192, 96), (257, 1536, 512)])
@pytest.mark.parametrize("xdt", [H.DTYPE_F32, H.DTYPE_BF16])
@pytest.mark.parametrize("fmt", ["q8_32", "q8_64", "q8_16", "q4_32", "q4_zeros_64", "fp8_64"])
def test_expanded_weight_equals_dequantized(be, monkeypatch, fmt, xdt, M, K, N):
    monkeypatch.setenv("LIGHTX2V_HIP_ROWS", "0")
    g, wf = int(fmt.split("_")[-1]), normal(4501 + N + K, N * K, 0.02).reshape(N, K)
    if fmt.startswith("q8"):
        q, s = O.q8_quantize(wf, N, K, g)
        w = be.weight_q8(q, s, N, K, g)
    elif fmt.startswith("q4"):
        c, s, z = O.q4_quantize_sym(wf, N, K, g)
        if "zeros" in fmt:
            z = z + (np.arange(z.size, dtype=np.float32).reshape(z.shape) % 3 - 1) * np.float32(0.5)
        w = be.weight_q4(O.q4_pack(c), s, z, N, K, g, packed=True)
    else:
        q, s = O.fp8_quantize(wf, N, K, g, True)
        w = be.weight_fp8(q, s, N, K, g)
    x, b = be.alloc((M + 1) * K, xdt), be.upload(normal(4503, N, 0.01))
    be.write(x, normal(4502, (M + 1) * K))
    if fmt == "fp8_64":
        be.set_fp8_act(H.FP8_ACT_BF16)
    try:
        for ydt in (H.DTYPE_BF16, H.DTYPE_F32):
            out = []
            for e in ("0", "1"):
                monkeypatch.setenv("LIGHTX2V_HIP_W16_EXPAND", e)
                v, names = _run(be, x, w, b, H.ACT_GELU_TANH, M, N, ydt)
                assert ("w16_expand" in names) == (e == "1"), names
                out.append(v)
            assert np.array_equal(u32(out[0]), u32(out[1]))
    finally:
        be.set_fp8_act(H.FP8_ACT_E4M3)


def _q8(be, seed, N, K):
    codes = (np.arange(N * K, dtype=np.uint32) * np.uint32(2654435761 + 2 * seed) >> np.uint32(24)).astype(np.uint8)
    return be.weight_q8(codes.view(np.int8), np.full(N * K // 32, 1e-3, np.float32), N, K, 32)


# 3 MB written out; 48 MiB and 128 KB, past the no-alloc scratch (its tiles give the same bits)
@pytest.mark.parametrize("M,K,N", [(300, 1024, 1536), (65, 8192, 3080)])
@pytest.mark.parametrize("xdt", [H.DTYPE_F32, H.DTYPE_BF16])
def test_expanded_without_allocations(be, monkeypatch, xdt, M, K, N):
    monkeypatch.setenv("LIGHTX2V_HIP_ROWS", "0")
    monkeypatch.setenv("LIGHTX2V_HIP_W16_EXPAND", "1")
    w, x, b = _q8(be, 1, N, K), be.alloc((M + 1) * K, xdt), be.upload(normal(4602, N, 0.01))
    be.write(x, normal(4601, (M + 1) * K))
    want, names = _run(be, x, w, b, H.ACT_NONE, M, N, H.DTYPE_F32)
    assert "w16_expand" in names
    y = be.alloc(M * N)
    for _ in range(2):
        be.write(y, np.full(M * N, np.nan, np.float32))
        be.linear_noalloc(x, 1, M, w, b, H.ACT_NONE, y, 0)
        assert np.array_equal(u32(be.download(y)), u32(want).ravel())


def test_expanded_in_graphs(monkeypatch):
    """A graph captured before there is a workspace for the written-out weight,
    and one captured after; then the context's workspaces outgrow what the
    graphs hold.  Every replay gives the eager bits, with eager work between."""
    monkeypatch.setenv("LIGHTX2V_HIP_ROWS", "0")
    monkeypatch.setenv("LIGHTX2V_HIP_W16_EXPAND", "1")
    be = H.HipBackend(0)
    try:
        M, K, N = 300, 1024, 1536
        w, x = _q8(be, 2, N, K), be.alloc(M * K, H.DTYPE_F32)
        xb = be.alloc(M * K, H.DTYPE_BF16)
        for buf in (x, xb):
            be.write(buf, normal(4701, M * K))
        y, y2, want = be.alloc(M * N), be.alloc(M * N), be.alloc(M * N)

        def capture(src, dst):
            be.graph_begin()
            be.linear(src, 0, M, w, None, H.ACT_GELU_TANH, dst, 0)
            return be.graph_end()

        graphs = [capture(xb, y)]  # no workspace yet: the tiles
        be.linear(x, 0, M, w, None, H.ACT_GELU_TANH, want, 0)
        ref = u32(be.download(want)).copy()
        graphs.append(capture(x, y2))
        big, bx, by = _q8(be, 3, 4096, 2048), be.alloc(900 * 2048, H.DTYPE_F32), be.alloc(900 * 4096)
        be.write(bx, normal(4702, 900 * 2048))
        for rep in range(3):
            be.linear(bx, 0, 900, big, None, H.ACT_NONE, by, 0)  # (the first of these grows both workspaces)
            for g, dst in zip(graphs, (y, y2)):
                be.write(dst, np.full(M * N, np.nan, np.float32))
                be.sync()
                g.launch()
                be.linear(bx, 0, 300 + 300 * rep, big, None, H.ACT_NONE, by, 0)
                assert np.array_equal(u32(be.download(dst)), ref), rep
        for g in graphs:
            g.free()
        be.linear(x, 0, M, w, None, H.ACT_GELU_TANH, want, 0)
        assert np.array_equal(u32(be.download(want)), ref)
    finally:
        be.close()
