"""int8 linears: where a pass that widens the weight costs more than it gains,
the launch widens inside its kernels, and the other way round. Each side's
result against the other's, forced."""
import numpy as np
import pytest

from test_gpu_kernels import synth

pytestmark = pytest.mark.gpu


# a wide weight and few rows (the pass reads and writes more than the tiles
# of either side take); the same from many rows on; few columns at long K; a
# ragged last tile row, on narrow tiles once the weight is widened
@pytest.mark.parametrize("rows,k,n,route", [
    (200, 4096, 24576, "qw_gemm_w8_store_q:split=2"), (700, 4096, 24576, "qw_gemm_w8_store_q:split=2"),
    (1152, 4096, 12288, "qw_gemm_w8_store_q"), (4119, 4096, 24576, "qw_gemm_bf16_store_mix:3x256+15x224"),
    (64, 12288, 3072, "qw_gemm_bf16_store_n1:split=8"),
    (4119, 12288, 4096, "qw_gemm_bf16_store_n1:split=8:from=4096 qw_gemm_bf16_store_q"),
    (9, 64, 8, "qw_gemm_bf16_store_n1"), (1000, 64, 2048, "qw_gemm_bf16_store_n1")])
def test_int8_linear_takes_the_faster_route(gpu, qd, oracle, monkeypatch, rows, k, n, route):
    w, q, s = gpu.new(n * k, qd.BF16), gpu.new(n * k, qd.I8), gpu.new(n, qd.F32)
    x = synth(oracle, rows * k, 61)
    gpu.check(qd.lib().qw_gpu_fill_normal_bf16(gpu.h, w.h, 0, n * k, 3, 4, 0.02, 0.0), "fill")
    gpu.check(qd.lib().h3_gpu_quantize_weight_int8(gpu.h, q.h, s.h, w.h, n, k), "quantize")
    out = gpu.new(rows * n, qd.BF16)
    gpu.linear(out, gpu.put(x), q, rows, k, n, wscale=s)
    assert gpu.route() == route
    gpu.submit()
    monkeypatch.setenv("QW_INT8_ROUTE", "widen" if "_w8_" in route else "w8")
    forced = qd.Gpu()
    try:
        other = forced.new(rows * n, qd.BF16)
        forced.linear(other, forced.put(x), q, rows, k, n, wscale=s)
        assert ("_w8_" in forced.route()) == ("_w8_" not in route)
        forced.submit()
        a, b = (oracle.bf16_to_f32(t.read()).reshape(rows, n) for t in (out, other))
    finally:
        forced.close()
    # two orders of one fp32 sum of k products differ by at most k 2^-24 of
    # sum |x w| <= |x| |w| each, and a bf16 rounding more
    xn = np.linalg.norm(oracle.bf16_to_f32(x).reshape(rows, k).astype(np.float64), axis=1)
    wn = np.array([np.linalg.norm(q.view(c * k, k).read().astype(np.float64)) for c in (0, n - 1)])
    wn = wn * s.read()[[0, n - 1]]
    for i, c in enumerate((0, n - 1)):
        tol = 2.0 ** -7 * np.abs(b[:, c]) + 2 * k * 2.0 ** -24 * xn * wn[i]
        assert (np.abs(a[:, c] - b[:, c]) <= tol).all()
    assert np.mean(a != b) < 0.02  # and elsewhere the sums mostly round alike
