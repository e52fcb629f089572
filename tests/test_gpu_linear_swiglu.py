"""The fused SwiGLU linear (qw_gpu_linear_swiglu) against the linear followed
by the separate SwiGLU pass, which have their own tests against the oracle.

Both take the same sums in the same order and silu of the same bf16 values,
rounded to bf16, so the results are the same bits."""
import ctypes as C

import numpy as np
import pytest

from conftest import ulp_diff

pytestmark = pytest.mark.gpu


def fused(gpu, qd, out, x, w, rows, k, F, ldc=None, **kw):
    h = lambda t: t.h if t is not None else None  # noqa: E731
    d = qd.LinearDesc(out.h, kw.get("out_offset", 0), ldc or F, x.h, 0, k, w.h,
                      h(kw.get("wscale")), h(kw.get("bias")), rows, k, 2 * F,
                      kw.get("epilogue", qd.LINEAR_STORE), *([None] * 2), 0, 0, *([None] * 4), 0,
                      0.0)
    return qd.lib().qw_gpu_linear_swiglu(gpu.h, C.byref(d))


# rows, k, F: narrow tiles of 64, 128 and 192 rows, whole and in pieces, ragged
# columns; the streaming rows; 256-row tiles above narrow ones, and alone
CASES = [(9, 64, 64, False), (100, 128, 200, True), (300, 1024, 448, False), (130, 4096, 256, True),
         (3, 256, 72, True), (8, 64, 128, False), (520, 2304, 4096, False), (2100, 64, 4224, True),
         (4119, 64, 3072, False)]


@pytest.mark.parametrize("route", ["bf16", "int8", "w8"])
@pytest.mark.parametrize("rows,k,F,bias", CASES)
def test_swiglu_linear_is_linear_then_swiglu(qd, oracle, monkeypatch, rows, k, F, bias, route):
    if route == "w8":
        monkeypatch.setenv("QW_INT8_ROUTE", "w8")
    gpu = qd.Gpu()
    try:
        x = gpu.put(oracle.fill_normal_bf16(rows * k, 7, 1, 1.0))
        w = gpu.put(oracle.fill_normal_bf16(2 * F * k, 7, 2, 1.5 / np.sqrt(k)))
        b = gpu.put(oracle.fill_normal_bf16(2 * F, 7, 3, 0.2)) if bias else None
        s = None
        if route != "bf16":
            q, s = gpu.new(2 * F * k, qd.I8), gpu.new(2 * F, qd.F32)
            gpu.check(qd.lib().h3_gpu_quantize_weight_int8(gpu.h, q.h, s.h, w.h, 2 * F, k), "q")
            w = q
        wide, two = gpu.new(rows * 2 * F, qd.BF16), gpu.new(rows * F, qd.BF16)
        gpu.linear(wide, x, w, rows, k, 2 * F, bias=b, wscale=s)
        gpu.check(qd.lib().qw_gpu_swiglu_bf16(gpu.h, two.h, wide.h, rows, F), "swiglu")
        pad = 0 if rows <= 8 else 8  # a strided output's gap stays untouched
        one = gpu.put(np.full(rows * (F + pad), 0x1234, np.uint16))
        gpu.check(fused(gpu, qd, one, x, w, rows, k, F, ldc=F + pad, bias=b, wscale=s), "fused")
        gpu.submit()
        got = one.read().reshape(rows, F + pad)
        assert (got[:, F:] == 0x1234).all()
        d = ulp_diff(np.ascontiguousarray(got[:, :F]).ravel(), two.read())
        assert d.max() == 0, (d.max(), np.mean(d != 0))
    finally:
        gpu.close()


# rows, k, F, narrow tiles allowed, the fused launch's kernels
ROUTES = [
    (4100, 256, 3072, True, "qw_gemm_bf16_swiglu_mix:3x224+18x192"),
    (2300, 256, 9224, True, "qw_gemm_bf16_swiglu_mix:2x256+8x224"),
    (2820, 64, 3072, False, "qw_gemm_bf16_swiglu_q:half=64"),
    (300, 4096, 1032, False, "qw_gemm_bf16_swiglu_q:split=2"),
    (2100, 64, 4224, True, "qw_gemm_bf16_swiglu_n2:from=1792 qw_gemm_bf16_swiglu_q"),
    (2900, 256, 3328, True, "qw_gemm_bf16_swiglu_n3:from=2304 qw_gemm_bf16_swiglu_q"),
    (1500, 256, 6664, True, "qw_gemm_bf16_swiglu_n4:from=1024 qw_gemm_bf16_swiglu_q"),
    (1000, 64, 4096, True, "qw_gemm_bf16_swiglu_n4"),
    (700, 4096, 1544, True, "qw_gemm_bf16_swiglu_n3:split=2"),
]


@pytest.mark.parametrize("rows,k,F,narrow,route", ROUTES)
def test_swiglu_linear_each_kernel(qd, monkeypatch, rows, k, F, narrow, route):
    """The same comparison on each bf16 kernel, by the route that ran: mixed
    tile heights, the half-tile and the split tail of wide tiles, narrow tiles
    below wide ones and alone; ragged columns among them."""
    if not narrow:
        monkeypatch.setenv("QW_GEMM_HALF_SMALL", "0")
    gpu = qd.Gpu()
    try:
        x, w, b = gpu.new(rows * k, qd.BF16), gpu.new(2 * F * k, qd.BF16), gpu.new(2 * F, qd.BF16)
        for i, (t, std) in enumerate(((x, 1.0), (w, 1.5 / np.sqrt(k)), (b, 0.2))):
            gpu.check(qd.lib().qw_gpu_fill_normal_bf16(gpu.h, t.h, 0, t.n, 7, i, std, 0.0), "fill")
        wide, two = gpu.new(rows * 2 * F, qd.BF16), gpu.new(rows * F, qd.BF16)
        gpu.linear(wide, x, w, rows, k, 2 * F, bias=b)
        gpu.check(qd.lib().qw_gpu_swiglu_bf16(gpu.h, two.h, wide.h, rows, F), "swiglu")
        one = gpu.put(np.full((rows + 1) * F, 0x1234, np.uint16))
        gpu.check(fused(gpu, qd, one, x, w, rows, k, F, bias=b), "fused")
        assert gpu.route() == route
        gpu.submit()
        got = one.read()
        assert np.array_equal(got[:rows * F], two.read()) and (got[rows * F:] == 0x1234).all()
    finally:
        gpu.close()


def test_swiglu_linear_every_gate(gpu, qd, oracle):
    """Each of the 65536 bf16 values as a gate (through the bias, weights 0),
    infinities and NaN among them: the separate pass's bits."""
    rows, k, F = 16, 64, 65536
    x, w = gpu.put(np.full(rows * k, 0x3F80, np.uint16)), gpu.put(np.zeros(2 * F * k, np.uint16))
    one = np.full(F, 0x3F80, np.uint16)
    b = gpu.put(np.concatenate([np.arange(F, dtype=np.uint32).astype(np.uint16), one]))
    wide, two, got = gpu.new(rows * 2 * F, qd.BF16), gpu.new(rows * F, qd.BF16), gpu.new(rows * F, qd.BF16)
    gpu.linear(wide, x, w, rows, k, 2 * F, bias=b)
    gpu.check(qd.lib().qw_gpu_swiglu_bf16(gpu.h, two.h, wide.h, rows, F), "swiglu")
    gpu.check(fused(gpu, qd, got, x, w, rows, k, F, bias=b), "fused")
    gpu.submit()
    a, r = got.read(), two.read()
    nan = np.isnan(oracle.bf16_to_f32(r))
    assert np.array_equal(np.isnan(oracle.bf16_to_f32(a)), nan)
    assert np.array_equal(a[~nan], r[~nan])


def test_swiglu_linear_gate_range(gpu, qd, oracle):
    """Gates over the whole bf16 range (x = I picks single weights): no
    overflow, and silu right to one bf16 ulp where the result is normal, up
    to the gates where e^-g overflows."""
    k = F = 64
    mags = np.geomspace(1e-30, 3e38, k * F // 2)
    g = np.concatenate([mags, -mags, ])
    g[:200] = np.linspace(-89.5, -80.0, 200)
    gb = oracle.f32_to_bf16(g.astype(np.float32)).reshape(F, k)
    up = oracle.f32_to_bf16(np.ones((F, k), np.float32))
    x = oracle.f32_to_bf16(np.eye(k, dtype=np.float32))
    out = gpu.new(k * F, qd.BF16)
    gpu.check(fused(gpu, qd, out, gpu.put(x), gpu.put(np.concatenate([gb, up])), k, k, F), "fused")
    gpu.submit()
    got = oracle.bf16_to_f32(out.read()).astype(np.float64).reshape(k, F).T
    v = oracle.bf16_to_f32(gb.ravel()).astype(np.float64).reshape(F, k)
    ref = np.where(v < -709, 0.0, v / (1.0 + np.exp(-np.maximum(v, -709))))
    # where e^-g overflows fp32 (g < -88.7) silu comes out as 0, as the
    # separate pass has it; one rounding to bf16 otherwise
    assert np.isfinite(got).all()
    live = v > -88.7
    assert (np.abs(got - ref)[live] <= 2.0 ** -8 * np.abs(ref)[live] + 2.0 ** -133).all()
    assert (np.abs(got)[~live] <= 1e-35).all()


@pytest.mark.parametrize("rows", [1, 8, 9])
@pytest.mark.parametrize("ldc,off", [(80, 0), (72, 16), (92, 4)])
def test_swiglu_linear_strided_output(gpu, qd, oracle, rows, ldc, off):
    """A strided output, or one at an offset, at any row count: the dense
    output's values (within the order of the sums), nothing beside them."""
    k, F = 128, 72
    x = gpu.put(oracle.fill_normal_bf16(rows * k, 7, 1, 1.0))
    w = gpu.put(oracle.fill_normal_bf16(2 * F * k, 7, 2, 1.5 / np.sqrt(k)))
    dense = gpu.new(rows * F, qd.BF16)
    gpu.check(fused(gpu, qd, dense, x, w, rows, k, F), "dense")
    out = gpu.put(np.full(off + rows * ldc, 0x1234, np.uint16))
    gpu.check(fused(gpu, qd, out, x, w, rows, k, F, ldc=ldc, out_offset=off), "strided")
    gpu.submit()
    got = out.read()
    assert (got[:off] == 0x1234).all()
    got = got[off:].reshape(rows, ldc)
    assert (got[:, F:] == 0x1234).all()
    a, b = oracle.bf16_to_f32(got[:, :F].ravel()), oracle.bf16_to_f32(dense.read())
    # g and u each a bf16 ulp apart at most where their sums' order differs
    # (silu passes at most 1.1 of g's step on), silu and the product one more
    # rounding each: 4 ulps of 2^-8, or of what a gate that cancels leaves
    assert (np.abs(a - b) <= 4 * 2.0 ** -8 * np.abs(b) + 2.0 ** -8).all()
    if rows == 9:
        assert np.array_equal(a, b)  # one kernel


def test_swiglu_linear_refusals(gpu, qd):
    F, k, rows = 64, 64, 16
    x, w, out = gpu.new(rows * k, qd.BF16), gpu.new(2 * F * k, qd.BF16), gpu.new(rows * F, qd.BF16)
    assert fused(gpu, qd, out, x, w, rows, k, F)
    assert not fused(gpu, qd, out, x, w, rows, k, F, ldc=F - 8)
    assert not fused(gpu, qd, out, x, w, rows + 1, k, F)
    assert not fused(gpu, qd, out, x, w, rows, k, F, epilogue=qd.LINEAR_GELU)
    assert not fused(gpu, qd, out, x, w, rows, k, F, epilogue=4)
    assert not fused(gpu, qd, out, x, w, 4, k, F, ldc=F - 8)
    assert not fused(gpu, qd, out, x, w, rows, k, F, ldc=F + 8)  # past the output's end
    for n in (4, rows):  # over the input, or its last elements, at any row count
        assert not fused(gpu, qd, x, x, w, n, k, F)
        both = gpu.new(2 * n * k, qd.BF16)
        assert not fused(gpu, qd, both.view(n * k - 4, n * F), both, w, n, k, F)
        assert fused(gpu, qd, both.view(n * k, n * F), both, w, n, k, F)
    d = qd.LinearDesc(out.h, 0, F, x.h, 0, k, w.h, None, None, rows, k, F, 4, None, None, 0, 0,
                      None, None, None, None, 0, 0.0)
    assert not qd.lib().qw_gpu_linear(gpu.h, C.byref(d))  # not an epilogue of qw_gpu_linear
    gpu.submit()
