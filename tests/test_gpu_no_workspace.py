"""Without memory for the runtime's workspaces (split partials, widened
copies) every linear and attention launch still runs, whole: the results of
the launches that have them, to the oracle's bars, with nothing allocated."""
import numpy as np
import pytest

import test_gpu_attention_split as A
import test_gpu_linear_narrow as N
from conftest import rel_l2
from test_gpu_kernels import assert_linear_close, synth

pytestmark = pytest.mark.gpu


@pytest.fixture
def bare(qd, monkeypatch):
    monkeypatch.setenv("QW_WORKSPACES", "0")
    gpu = qd.Gpu()
    yield gpu
    gpu.close()


# what each runs as with workspaces: narrow tiles in pieces, narrow tiles below
# wide ones, mixed heights, narrow tiles in pieces below wide ones, wide tiles
# in pieces
@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("rows,k,n", [(63, 8192, 264), (320, 3072, 1024), (2305, 1024, 7176),
                                      (4315, 512, 3072), (4400, 4096, 4096), (1152, 12288, 4096)])
def test_linear_without_workspace(bare, qd, oracle, rows, k, n, int8):
    x, w, s, b, lin, mag = N._operands(bare, oracle, rows, k, n, int8)
    out = bare.new(rows * n, qd.BF16)
    before = bare.stats().allocated_bytes
    bare.linear(out, x, w, rows, k, n, bias=b, wscale=s)
    assert "split=" not in bare.route() and ("_w8_" in bare.route()) == int8
    bare.submit()
    assert bare.stats().allocated_bytes == before
    assert_linear_close(oracle, out.read(), lin, mag)


@pytest.mark.parametrize("rows,heads", [(1000, 1), (2100, 32)])  # few blocks; past full rounds
def test_attention_without_workspace(bare, gpu, qd, oracle, rows, heads):
    q, k, v = (synth(oracle, rows * heads * 128, 200 + i) for i in range(3))
    want = A.run(gpu, qd, q, k, v, 1, rows, rows, heads)
    H = heads * 128
    qt, kt, vt, out = bare.put(q), bare.put(k), bare.put(v), bare.new(rows * H, qd.BF16)
    before = bare.stats().allocated_bytes
    assert "split=" in gpu.route()
    bare.attention(out, qt, kt, vt, 1, rows, rows, heads, H, H, H, H)
    assert "split=" not in bare.route()
    bare.submit()
    assert bare.stats().allocated_bytes == before
    assert rel_l2(oracle.bf16_to_f32(out.read()), oracle.bf16_to_f32(want.ravel())) < 5e-3
