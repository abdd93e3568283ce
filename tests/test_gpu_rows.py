"""The few-rows linear (csrc/k_gemm_rows.hip: FP8 up to 64 rows, the others up to
256) against the tile kernels on the same operands (LIGHTX2V_HIP_ROWS=0), for
every weight format and activation / output type that takes it, at its edges:
one row, whole and ragged 32-row blocks, one to four 64-row workgroups, whole
and ragged 32-channel blocks, K below, at and past the eight waves' first
steps, row offsets.  And which of the ways a call takes.

Both sides contract the same e4m3 / bf16 operands and differ in the order of
their f32 sums (and in the point where a group's scale enters): FP8_TIGHT
(the fp8 MFMA's own dot error, 1.5e-5) and W16_TIGHT bound that for f32
outputs.  A bf16 output may then round to the neighbouring value: within one
bf16 step of the f32 one.  MX e4m3 output equals quantize_mx of the kernel's
own f32 output bit for bit.
"""

import numpy as np
import pytest

import lightx2v_hip as H
import oracle as O
from helpers import FP8_TIGHT, W16_TIGHT, assert_close, normal, oracle_w16, u32

pytestmark = pytest.mark.gpu

SHAPES = [(1, 64, 32), (17, 1536, 96), (32, 128, 1000), (33, 1152, 64), (64, 2304, 33)]


def _weight(be, fmt, N, K):
    wf = normal(4001 + N + K, N * K, 0.02).reshape(N, K)
    if fmt == "native":
        return be.weight(wf, N, K), wf
    if fmt.startswith("q8"):
        g = int(fmt[3:])
        q, s = O.q8_quantize(wf, N, K, g)
        return be.weight_q8(q, s, N, K, g), O.q8_dequantize(q, s, N, K, g)
    if fmt.startswith("q4"):
        g = int(fmt.split("_")[-1])
        c, s, z = O.q4_quantize_sym(wf, N, K, g)
        if "zeros" in fmt:
            z = z + (np.arange(z.size, dtype=np.float32).reshape(z.shape) % 3 - 1) * np.float32(0.5)
        return be.weight_q4(O.q4_pack(c), s, z, N, K, g, packed=True), O.q4_dequantize(c, s, z, N, K, g)
    g = K if fmt == "fp8" else int(fmt[4:])
    q, s = O.fp8_quantize(wf, N, K, g, True)
    return be.weight_fp8(q, s, N, K, g), O.fp8_dequantize(q, s, N, K, g)


def _linear(be, monkeypatch, few, x, row, M, w, b, act, y, y_row):
    monkeypatch.setenv("LIGHTX2V_HIP_ROWS", "256" if few else "0")
    be.profile_reset()
    be.profile_enable(True)
    try:
        be.linear(x, row, M, w, b, act, y, y_row)
        names = [k for k in be.profile_stats() if k.startswith("gemm")]
    finally:
        be.profile_enable(False)
        be.profile_reset()
    assert [".rows" in k for k in names] == [few], names


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("xdt", [H.DTYPE_F32, H.DTYPE_BF16])
@pytest.mark.parametrize("fmt", ["native", "q8_32", "q8_64", "q8_16", "q4_32", "q4_zeros_32", "fp8_64", "fp8", "fp8_128"])
def test_rows_vs_tiles(be, monkeypatch, fmt, xdt, M, K, N):
    if fmt == "fp8_128" and K % 128:
        pytest.skip("group 128 needs cols % 128 == 0")
    w, wd = _weight(be, fmt, N, K)
    x, b = normal(4101 + M, (M + 3) * K).reshape(M + 3, K), normal(4102, N, 0.01)
    xb, bb = be.alloc(x.size, xdt), be.upload(b)
    be.write(xb, x)
    fp8 = fmt in ("fp8", "fp8_128") or (fmt == "fp8_64" and K == 64)  # contracted on the fp8 MFMA
    out = []
    for few in (False, True):
        y = be.alloc((M + 2) * N, H.DTYPE_F32)
        be.write(y, np.full((M + 2) * N, np.nan, np.float32))
        _linear(be, monkeypatch, few, xb, 3, M, w, bb, H.ACT_GELU_TANH, y, 1)
        v = be.download(y).reshape(M + 2, N)
        assert np.isnan(v[0]).all() and np.isnan(v[-1]).all()  # nothing written outside the rows
        out.append(v[1:-1])
    assert_close(out[1], out[0], *(FP8_TIGHT if fp8 else W16_TIGHT), what=f"{fmt} rows vs tiles")
    if not fp8:
        assert_close(out[1], oracle_w16(x[3:], wd, b, 1), *W16_TIGHT, what=f"{fmt} rows vs oracle")
    y16 = be.alloc(M * N, H.DTYPE_BF16)
    _linear(be, monkeypatch, True, xb, 3, M, w, bb, H.ACT_GELU_TANH, y16, 0)
    assert np.array_equal(u32(be.download(y16)), u32(O.bf16_round(out[1]).ravel()))


@pytest.mark.parametrize("M,K,N", [(65, 1152, 33), (128, 192, 64), (129, 1536, 96), (256, 64, 1000)])
@pytest.mark.parametrize("xdt", [H.DTYPE_F32, H.DTYPE_BF16])
@pytest.mark.parametrize("fmt", ["native", "q8_32", "q4_32", "q4_zeros_32", "fp8_64"])
def test_rows_past_one_workgroup(be, monkeypatch, fmt, xdt, M, K, N):
    """More than 64 rows: workgroups of 64, the last one ragged."""
    if fmt == "fp8_64" and K == 64:
        pytest.skip("one group per channel: the fp8 MFMA")
    w, wd = _weight(be, fmt, N, K)
    x, b = normal(4401 + M, (M + 3) * K).reshape(M + 3, K), normal(4402, N, 0.01)
    xb, bb = be.alloc(x.size, xdt), be.upload(b)
    be.write(xb, x)
    out = []
    for few in (False, True):
        y = be.alloc((M + 2) * N, H.DTYPE_F32)
        be.write(y, np.full((M + 2) * N, np.nan, np.float32))
        _linear(be, monkeypatch, few, xb, 3, M, w, bb, H.ACT_GELU_TANH, y, 1)
        v = be.download(y).reshape(M + 2, N)
        assert np.isnan(v[0]).all() and np.isnan(v[-1]).all()
        out.append(v[1:-1])
    assert_close(out[1], out[0], *W16_TIGHT, what=f"{fmt} rows vs tiles")
    assert_close(out[1], oracle_w16(x[3:], wd, b, 1), *W16_TIGHT, what=f"{fmt} rows vs oracle")


@pytest.mark.parametrize("M,K,N", [(1, 128, 32), (17, 1536, 96), (33, 1152, 64), (64, 2304, 1024)])
@pytest.mark.parametrize("fmt", ["fp8", "fp8_128"])
@pytest.mark.parametrize("x_mx", [False, True])
def test_rows_fp8_quantized_operands(be, monkeypatch, x_mx, fmt, M, K, N):
    """Per-token and MX e4m3 input (MX from row 16 on), f32 and MX output."""
    w, _ = _weight(be, fmt, N, K)
    r0 = 16
    xb, bb = be.upload(normal(4201 + M, (M + r0) * K)), be.upload(normal(4202, N, 0.01))
    xq = be.alloc_mx(M + r0, K) if x_mx else be.alloc_e4m3(M + r0, K)
    (be.quantize_mx if x_mx else be.quantize_act)(xb, 0, M + r0, xq)
    out = []
    for few in (False, True):
        y = be.alloc(M * N, H.DTYPE_F32)
        _linear(be, monkeypatch, few, xq, r0, M, w, bb, H.ACT_NONE, y, 0)
        out.append(be.download(y).reshape(M, N))
    assert_close(out[1], out[0], *FP8_TIGHT, what=f"{fmt} rows vs tiles")
    ym, ref = be.alloc_mx(M, N), be.alloc_mx(M, N)
    _linear(be, monkeypatch, True, xq, r0, M, w, bb, H.ACT_NONE, ym, 0)
    be.quantize_mx(be.upload(out[1]), 0, M, ref)
    for a, c in zip(be.download_mx(ym, M, N), be.download_mx(ref, M, N)):
        assert np.array_equal(a, c)


@pytest.mark.parametrize("hdt", [H.DTYPE_F32, H.DTYPE_BF16])
@pytest.mark.parametrize("fmt", ["fp8", "fp8_128"])
def test_rows_residual_equals_pair(be, monkeypatch, fmt, hdt):
    """linear_residual on few rows == linear, then gate_residual, bit for bit."""
    monkeypatch.setenv("LIGHTX2V_HIP_ROWS", "64")
    M, K, N = 40, 1536, 96
    w, _ = _weight(be, fmt, N, K)
    xb, bb, h0 = be.upload(normal(4301, M * K)), be.upload(normal(4302, N, 0.01)), normal(4303, M * N)
    mods = be.upload(normal(4304, 2 * N))
    h1, h2, y = (be.alloc(M * N, hdt) for _ in range(3))
    be.write(h1, h0)
    be.write(h2, h0)
    be.linear_residual(xb, 0, M, w, bb, H.ACT_NONE, h1, 0, mods, 1)
    be.linear(xb, 0, M, w, bb, H.ACT_NONE, y, 0)
    be.gate_residual(h2, y, M, N, mods, 1)
    assert np.array_equal(u32(be.download(h1)), u32(be.download(h2)))


# Calls where one way is at least 1.3 times the next (us, rows / tiles or rows / written out / tiles)
@pytest.mark.parametrize("fmt,xdt,M,K,N,way", [
    ("q8", "bf16", 17, 1536, 1536, "rows"),       # 9 / 13 / 23
    ("q4", "f32", 17, 3072, 3072, "rows"),        # 16 / 30 / 46
    ("q8", "bf16", 200, 14336, 3072, "written"),  # 147 / 77 / 197
    ("q4", "f32", 64, 14336, 1536, "written"),    # 129 / 73 / 189
    ("q8", "f32", 256, 8960, 1536, "written"),    # 82 / 52 / 128
    ("q8", "bf16", 128, 1536, 8960, "tiles"),     # 35 / 30 / 23
    ("native", "f32", 1, 1984, 9000, "tiles"),    # 20 / 13
    ("native", "bf16", 64, 1536, 8960, "tiles"),  # 24 / 8
    ("fp8", "bf16", 17, 8960, 1536, "rows"),      # 15 / 25 (the quantization aside)
    ("fp8", "e4m3", 33, 14336, 3072, "tiles"),    # 36 / 29
    ("fp8", "mx", 33, 1536, 8960, "tiles"),       # 16 / 10
    ("fp8_128", "bf16", 64, 1536, 8960, "tiles"),  # 22 / 14
    ("fp8_128", "mx", 64, 1536, 8960, "tiles"),   # 19 / 11
])
def test_the_faster_kernel_is_taken(be, monkeypatch, fmt, xdt, M, K, N, way):
    for k in ("ROWS", "W16_EXPAND", "W16_CFG", "FP8_CFG", "BF16_CFG", "FP8_SPLITK"):
        monkeypatch.delenv(f"LIGHTX2V_HIP_{k}", raising=False)
    codes = (np.arange(N * K, dtype=np.uint32) * np.uint32(2654435761) >> np.uint32(24)).astype(np.uint8)
    if fmt == "native":
        w = be.weight((codes.astype(np.float32) - 128) * np.float32(1e-3), N, K)
    elif fmt == "q8":
        w = be.weight_q8(codes.view(np.int8), np.full(N * K // 32, 1e-3, np.float32), N, K, 32)
    elif fmt == "q4":
        w = be.weight_q4(codes[:N * K // 2], np.full(N * K // 32, 1e-2, np.float32), np.full(N * K // 32, 8, np.float32),
                         N, K, 32, packed=True)
    else:
        g = K if fmt == "fp8" else 128
        codes = codes & 0xBF
        w = be.weight_fp8(np.where((codes & 0x78) == 0, codes & 0x80, codes).astype(np.uint8),
                          np.full(N * K // g, 1e-2, np.float32), N, K, g)
    x, y = be.alloc(M * K, H.DTYPE_F32 if xdt == "f32" else H.DTYPE_BF16), be.alloc(M * N, H.DTYPE_BF16)
    if xdt in ("mx", "e4m3"):
        x = be.alloc_mx(M, K) if xdt == "mx" else be.alloc_e4m3(M, K)
    be.profile_reset()
    be.profile_enable(True)
    try:
        be.linear(x, 0, M, w, None, H.ACT_NONE, y, 0)
        names = list(be.profile_stats())
    finally:
        be.profile_enable(False)
        be.profile_reset()
    got = "rows" if any(".rows" in k for k in names) else "written" if "w16_expand" in names else "tiles"
    assert got == way, names
