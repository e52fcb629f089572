"""The fused q|k|v projection with k and v in tensors of their own, against
the same projection beside q, bit for bit; and a block's K/V outputs, which
are those tensors where they can be."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_kernels import synth

pytestmark = pytest.mark.gpu


# narrow tiles in pieces, whole (int8 widened) and below wide ones; 256-row
# tiles wide and narrow; mixed tile heights of 224 and 192 and of 256 and 224
# rows; a table too short for the fused epilogue
@pytest.mark.parametrize("rows,k,heads,int8,rope_rows,route", [
    (70, 2048, 2, False, 200, "qw_gemm_bf16_qkn_n1:split=3"),
    (320, 256, 24, True, 320, "qw_gemm_bf16_qkn_n2"),
    (11400, 512, 4, False, 5700, "qw_gemm_bf16_qkn_n1:from=10752 qw_gemm_bf16_qkn_q"),
    (4119, 512, 10, False, 4119, "qw_gemm_bf16_qkn_q"),
    (3000, 192, 12, False, 1500, "qw_gemm_bf16_qkn_n4"),
    (4100, 192, 16, False, 4100, "qw_gemm_bf16_qkn_mix:3x224+18x192"),
    (2300, 256, 48, True, 1150, "qw_gemm_bf16_qkn_mix:2x256+8x224"),
    (300, 128, 2, False, 100, "qw_gemm_bf16_store_n1")])
def test_qkv_linear_outputs(gpu, qd, oracle, rows, k, heads, int8, rope_rows, route):
    H = heads * 128
    n = 3 * H
    x = gpu.put(synth(oracle, rows * k, 91))
    w = gpu.put(synth(oracle, n * k, 92, 0.05))
    s = None
    if int8:
        q, s = gpu.new(n * k, qd.I8), gpu.new(n, qd.F32)
        gpu.check(qd.lib().h3_gpu_quantize_weight_int8(gpu.h, q.h, s.h, w.h, n, k), "q")
        w = q
    ang = np.random.default_rng(9).uniform(-3, 3, (rope_rows, 64)).astype(np.float32)
    nq, nk = gpu.put(synth(oracle, 128, 34, 0.1)), gpu.put(synth(oracle, 128, 35, 0.1))
    ct, st = gpu.put(np.cos(ang)), gpu.put(np.sin(ang))
    ref, out = gpu.new(rows * n, qd.BF16), gpu.new(rows * n, qd.BF16)
    gpu.linear(ref, x, w, rows, k, n, wscale=s, epilogue=qd.LINEAR_QKNORM,
               qknorm=(nq, nk, ct, st, rope_rows, 1e-6))
    at = 8 * H  # rows before and after the written ones stay untouched
    kt, vt = (gpu.put(np.full((rows + 16) * H, 0x1234, np.uint16)) for _ in range(2))
    d = qd.LinearDesc(out.h, 0, n, x.h, 0, k, w.h, s.h if s else None, None, rows, k, n,
                      qd.LINEAR_QKNORM, None, None, 0, 0, nq.h, nk.h, ct.h, st.h, rope_rows, 1e-6)
    gpu.check(qd.lib().qw_gpu_qkv_linear(gpu.h, C.byref(d), kt.h, vt.h, at), "qkv")
    assert gpu.route() == route
    gpu.submit()
    want = ref.read().reshape(rows, 3, H)
    assert np.array_equal(out.read().reshape(rows, 3, H)[:, 0], want[:, 0])
    for i, t in ((1, kt), (2, vt)):
        got = t.read().reshape(rows + 16, H)
        assert (got[:8] == 0x1234).all() and (got[rows + 8:] == 0x1234).all()
        assert np.array_equal(got[8:rows + 8], want[:, i])
    d.epilogue = qd.LINEAR_STORE
    assert not qd.lib().qw_gpu_qkv_linear(gpu.h, C.byref(d), kt.h, vt.h, at)
    d.epilogue = qd.LINEAR_QKNORM
    assert not qd.lib().qw_gpu_qkv_linear(gpu.h, C.byref(d), kt.h, vt.h, at + 9 * H)
    gpu.submit()


@pytest.mark.parametrize("rope_rows", [100, 200])  # copied out, and stored by the epilogue
def test_qkv_linear_refusals(gpu, qd, rope_rows):
    """What k and v may be does not depend on the RoPE table's length: apart,
    16-byte aligned, and clear of the input and the output."""
    rows, k, H = 24, 512, 128
    n = 3 * H
    x, w, out = (gpu.new(m, qd.BF16) for m in (rows * k + rows * H, n * k, rows * n + rows * H))
    nq, ct = gpu.new(128, qd.BF16), gpu.new(rope_rows * 64, qd.F32)
    kv = gpu.new(4 * rows * H, qd.BF16)
    size = rows * H
    d = qd.LinearDesc(out.h, 0, n, x.h, 0, k, w.h, None, None, rows, k, n, qd.LINEAR_QKNORM, None,
                      None, 0, 0, nq.h, nq.h, ct.h, ct.h, rope_rows, 1e-6)
    call = lambda a, b, off=0: qd.lib().qw_gpu_qkv_linear(gpu.h, C.byref(d), a.h, b.h, off)  # noqa: E731
    assert call(kv, kv.view(size, size))
    assert call(kv.view(size, size), kv)
    assert call(out.view(rows * n, size), x.view(rows * k, size))
    assert not call(kv, kv)
    assert not call(kv, kv.view(size - 8, size)) and not call(kv.view(size - 8, size), kv)
    for off in (1, 2, 4):
        assert not call(kv, kv.view(2 * size, 2 * size), off)
        assert not call(kv.view(off, size), kv.view(2 * size, size))
        assert not call(kv, kv.view(2 * size + off, size))
    assert call(kv, kv.view(2 * size, 2 * size), 8)
    assert not call(out.view(rows * n - 8, size), kv) and not call(kv, out.view(0, size))
    assert not call(x.view(rows * k - 8, size), kv) and not call(kv, x.view(0, size))
    gpu.submit()


def test_block_kv_outputs(gpu, qd, oracle):
    """K/V outputs that attention reads in place (aligned, apart), and ones it
    cannot (at an odd element, or one tensor for both): the same hidden state
    and the same rows."""
    T, R = 16, 80
    cfg = dict(hidden=256, heads=2, mlp_width=512, text_dim=256, z_dim=64, layers=1, mlp_act=0,
               adaln_shift=0, has_bias=0, text_causal=1, int8_weights=0)
    dit = qd.Dit(gpu, cfg, 5)
    H = 256
    x, mod = synth(oracle, R * H, 1), synth(oracle, 2 * 4 * H, 2, 0.2)
    cos, sin = oracle.rope_tables(T, 8, 8)
    ct, st, mt = gpu.put(cos), gpu.put(sin), gpu.put(mod)
    rm = gpu.put((np.arange(R) < T).astype(np.uint32))
    res = []
    for form in ("none", "aligned", "odd", "one"):
        h = gpu.put(x)
        a, b = gpu.new(R * H + 8, qd.BF16), gpu.new(R * H + 8, qd.BF16)
        kv = {"none": (None, None), "aligned": (a, b), "one": (a, a),
              "odd": (a.view(2, R * H), b.view(2, R * H))}[form]
        dit.block(0, h, mt, ct, st, rm, R, T, k_out=kv[0], v_out=kv[1])
        gpu.submit()
        res.append((h.read(), [t.read()[:R * H] if t else None for t in kv]))
    dit.close()
    for h, _ in res[1:]:
        assert np.array_equal(h, res[0][0])
    assert np.array_equal(res[1][1][0], res[2][1][0])
    assert np.array_equal(res[1][1][1], res[2][1][1])
    assert np.array_equal(res[3][1][0], res[1][1][1])  # v after k, in one tensor
