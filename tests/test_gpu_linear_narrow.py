"""Narrow tiles (64-256 rows x 128 columns, in k-range pieces where tiles are
few) against the oracle, at the edges of their tiles, columns and k-ranges,
and the wide tiles at shapes that narrow ones would otherwise take."""
import numpy as np
import pytest

import test_gpu_kernels as K
from test_gpu_kernels import assert_gelu_close, assert_linear_close, bf16_neighbours, synth, ulp_diff

pytestmark = pytest.mark.gpu

# rows, k, n: one k-slice; fewer slices than stages; ragged columns; a piece
# per few slices; one and two rows past a tile; each tile height; each with a
# last tile row on narrow tiles below wide ones (4119 and 2305 rows)
SHAPES = [(9, 64, 8), (9, 4096, 8), (65, 128, 136), (63, 8192, 264), (257, 512, 1032),
          (700, 64, 3072), (320, 1024, 12288), (640, 128, 9216), (700, 4096, 3072),
          (1100, 2048, 1032), (300, 8192, 1544), (577, 320, 9216), (4119, 512, 4096),
          (2305, 1024, 7176)]


def _operands(gpu, oracle, rows, k, n, int8):
    x, w = synth(oracle, rows * k, 71), synth(oracle, n * k, 72, 0.02)
    b = synth(oracle, n, 73, 0.02)
    if int8:
        q, s = oracle.quantize_int8_rows(w, n, k)
        lin = oracle.linear_i8(x, q, s, b, rows, k, n)
        wt, st = gpu.put(q), gpu.put(s)
    else:
        lin, wt, st = oracle.linear(x, w, b, rows, k, n), gpu.put(w), None
    mag = oracle.bf16_to_f32(oracle.linear(x & np.uint16(0x7FFF), w & np.uint16(0x7FFF), None,
                                           rows, k, n)).ravel()
    return gpu.put(x), wt, st, gpu.put(b), lin.ravel(), mag


@pytest.mark.parametrize("rows,k,n", SHAPES)
def test_narrow_tiles_store_gelu_gate(gpu, qd, oracle, rows, k, n):
    int8 = (rows + n) % 3 == 0
    xt, wt, st, bt, lin, mag = _operands(gpu, oracle, rows, k, n, int8)
    pad = 8  # the gap between output rows and the rows past the last stay untouched
    out = gpu.put(np.full((rows + 1) * (n + pad), 0x1234, np.uint16))
    for _ in range(2):  # the pieces' counters are back at zero for a second call
        gpu.linear(out, xt, wt, rows, k, n, bias=bt, wscale=st, ldc=n + pad)
    gpu.submit()
    got = out.read().reshape(rows + 1, n + pad)
    assert (got[:, n:] == 0x1234).all() and (got[rows] == 0x1234).all()
    assert_linear_close(oracle, np.ascontiguousarray(got[:rows, :n]).ravel(), lin, mag)
    if rows <= 8 or n > 4096:
        return
    out = gpu.new(rows * n, qd.BF16)
    gpu.linear(out, xt, wt, rows, k, n, bias=bt, wscale=st, epilogue=qd.LINEAR_GELU)
    gpu.submit()
    assert_gelu_close(oracle, out.read(), lin, mag)
    mod, h0 = synth(oracle, 2 * 6 * n, 74, 0.5), synth(oracle, rows * n, 75)
    rm = (np.arange(rows) % 3 == 1).astype(np.uint32)
    out = gpu.put(h0)
    gpu.linear(out, xt, wt, rows, k, n, bias=bt, wscale=st, epilogue=qd.LINEAR_GATE,
               modulation=gpu.put(mod), row_map=gpu.put(rm), slots=6, gate_slot=2)
    gpu.submit()
    best = None  # the gate of y or of a bf16 neighbour of y, within one ulp
    for yv in (lin,) + bf16_neighbours(lin):
        want = np.empty(rows * n, np.uint16)
        oracle.lib().qo_gate(want, h0, np.ascontiguousarray(yv), mod, rm, rows, n, 6, 2)
        d = ulp_diff(out.read(), want)
        best = d if best is None else np.minimum(best, d)
    assert best.max() <= 1, best.max()


@pytest.mark.parametrize("rows,k,heads,route", [
    (70, 512, 2, "qw_gemm_bf16_qkn_n1"), (320, 3072, 4, "qw_gemm_bf16_qkn_n1:split=4"),
    (640, 256, 24, "qw_gemm_bf16_qkn_n4"), (4119, 512, 10, "qw_gemm_bf16_qkn_q"),
    (11400, 512, 4, "qw_gemm_bf16_qkn_n1:from=10752 qw_gemm_bf16_qkn_q"),
    (2900, 256, 17, "qw_gemm_bf16_qkn_n2:from=2304 qw_gemm_bf16_qkn_q")])
def test_narrow_tiles_qknorm(gpu, qd, oracle, rows, k, heads, route):
    """The q/k norm + RoPE epilogue bit for bit against the plain linear and
    the standalone kernel (the same tiles, whatever the epilogue): rows past
    a table's end wrap, and the table rows of narrow tiles below wide ones
    start where those end."""
    n = 3 * heads * 128
    xt, wt, _, bt, _, _ = _operands(gpu, oracle, rows, k, n, False)
    rope_rows = 200
    ang = np.random.default_rng(9).uniform(-3, 3, (rope_rows, 64)).astype(np.float32)
    ct, st = gpu.put(np.cos(ang)), gpu.put(np.sin(ang))
    nq, nk = gpu.put(synth(oracle, 128, 34, 0.1)), gpu.put(synth(oracle, 128, 35, 0.1))
    fused, ref = gpu.new(rows * n, qd.BF16), gpu.new(rows * n, qd.BF16)
    gpu.linear(fused, xt, wt, rows, k, n, bias=bt, epilogue=qd.LINEAR_QKNORM,
               qknorm=(nq, nk, ct, st, rope_rows, 1e-6))
    assert gpu.route() == route
    gpu.linear(ref, xt, wt, rows, k, n, bias=bt)
    gpu.check(qd.lib().qw_gpu_qk_norm_rope_bf16(gpu.h, ref.h, rows, heads, n, n // 3, nq.h, nk.h,
                                                 ct.h, st.h, rope_rows, 1e-6), "qk")
    gpu.submit()
    assert np.array_equal(fused.read(), ref.read())


# columns: in 8 tile columns 184 tiles of 192 rows fit a round, in 12 the 240
# of 224 rows do
@pytest.mark.parametrize("n,int8,tiles", [(1800, False, "0x224+23x192"), (1784, True, "0x224+23x192"),
                                          (3000, False, "0x256+20x224"), (2984, True, "0x256+20x224")])
def test_wide_low_tiles(qd, oracle, monkeypatch, n, int8, tiles):
    """test_linear_224_row_tiles_ragged_cols on tiles of 192 and 224 rows,
    with narrow tiles off; int8 weights widened by a pass."""
    monkeypatch.setenv("QW_GEMM_HALF_SMALL", "0")
    monkeypatch.setenv("QW_INT8_ROUTE", "widen")
    gpu = qd.Gpu()
    try:
        K.test_linear_224_row_tiles_ragged_cols(gpu, qd, oracle, n, int8)
        assert gpu.route() == "qw_gemm_bf16_store_mix:" + tiles
    finally:
        gpu.close()


@pytest.mark.parametrize("epi", ["store", "gelu", "gate"])
def test_wide_tile_walk(qd, oracle, monkeypatch, epi):
    """test_linear_tile_walk with narrow tiles off: the last 33 of its 289
    tiles run as 66 half tiles."""
    monkeypatch.setenv("QW_GEMM_HALF_SMALL", "0")
    gpu = qd.Gpu()
    try:
        K.test_linear_tile_walk(gpu, qd, oracle, epi)
        assert gpu.route() == f"qw_gemm_bf16_{epi}_q:half=66"
    finally:
        gpu.close()


def test_wide_half_tiles_qknorm(qd, oracle, monkeypatch):
    """The q/k norm + RoPE epilogue on the half tiles that end a tile walk
    (270 tiles: the last 14 as 28), with narrow tiles off."""
    monkeypatch.setenv("QW_GEMM_HALF_SMALL", "0")
    gpu = qd.Gpu()
    try:
        K.test_linear_qknorm_epilogue_bit_identical(gpu, qd, oracle, 11400, False, 11400, 512)
        assert gpu.route() == "qw_gemm_bf16_store_q:half=28"  # the plain linear it ends with
    finally:
        gpu.close()


@pytest.mark.parametrize("case", K.SPLIT_CASES)
def test_wide_split_tiles(qd, oracle, monkeypatch, case):
    """The shapes of test_linear_split_tiles with narrow tiles off, so that
    the wide tiles' split pieces run them."""
    monkeypatch.setenv("QW_GEMM_HALF_SMALL", "0")
    gpu = qd.Gpu()
    try:
        K.test_linear_split_tiles(gpu, qd, oracle, *case)
        assert "_q:split=" in gpu.route()
    finally:
        gpu.close()


def test_narrow_int8_weight_past_a_buffer_widened(gpu, qd, oracle):
    """An int8 weight of over 2^30 elements, whose widened copy would pass the 2
    GiB that a buffer covers: a launch that narrow tiles would suit stays on
    the kernels that widen inside."""
    rows, k, n, step = 60, 33792, 33024, 4128
    x = synth(oracle, rows * k, 81)
    xt, w, q, s = gpu.put(x), gpu.new(step * k, qd.BF16), gpu.new(n * k, qd.I8), gpu.new(n, qd.F32)
    for r in range(0, n, step):
        gpu.check(qd.lib().qw_gpu_fill_normal_bf16(gpu.h, w.h, 0, step * k, 3, r, 0.02, 0.0), "fill")
        qv, sv = q.view(r * k, step * k), s.view(r, step)
        gpu.check(qd.lib().h3_gpu_quantize_weight_int8(gpu.h, qv.h, sv.h, w.h, step, k), "quantize")
    out = gpu.new(rows * n, qd.BF16)
    gpu.linear(out, xt, q, rows, k, n, wscale=s)
    gpu.submit()
    got = out.read().reshape(rows, n)
    for c in (0, 8, 16384, n - 16):  # 8 columns at a time
        qc = q.view(c * k, 8 * k).read()
        lin = oracle.linear_i8(x, qc, s.view(c, 8).read(), None, rows, k, 8)
        mag = np.abs(oracle.bf16_to_f32(x).reshape(rows, k)) @ np.abs(qc.reshape(8, k).T.astype(np.float32))
        assert_linear_close(oracle, np.ascontiguousarray(got[:, c:c + 8]).ravel(), lin.ravel(),
                            (mag * s.view(c, 8).read()).ravel())
