"""Attention launches whose blocks are cut along the keys (few query blocks,
or a partly filled last round of them): against the oracle, and a row's
result against the same row's in a launch that differs in the other rows."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_kernels import synth

pytestmark = pytest.mark.gpu


def run(gpu, qd, q, k, v, batch, q_rows, kv_rows, heads, **kw):
    H = heads * 128
    out = gpu.put(np.full(batch * q_rows * H, 0x7FC0, np.uint16))  # NaN: every row is written
    for _ in range(2):  # the counters are back at zero for a second call
        gpu.attention(out, gpu.put(q), gpu.put(k), gpu.put(v), batch, q_rows, kv_rows, heads, H, H,
                      H, H, **kw)
    gpu.submit()
    return out.read().reshape(batch, q_rows, H)


# rows, heads, text, causal, batch: few blocks in up to 8 pieces (text rows
# see only the first ones); 32 blocks of 256 past one full round of them, and
# ragged; two batches with leading blocks that are all text, the round counted
# in the others; and two that run whole (few keys; nearly full last rounds)
@pytest.mark.parametrize("rows,heads,text,causal,batch,route", [
    (1152, 3, 128, 0, 1, "qw_attention_w4_split_bf16:split=3"),
    (1000, 1, 300, 1, 1, "qw_attention_w4_split_bf16:split=4"),
    (2100, 32, 23, 1, 1, "qw_attention_split_bf16:split=5:from=256"),
    (2100, 20, 512, 0, 2, "qw_attention_split_bf16:split=5:from=330"),
    (513, 2, 0, 0, 1, "qw_attention_w4_bf16"), (2304, 17, 512, 0, 2, "qw_attention_bf16")])
def test_split_attention_oracle(gpu, qd, oracle, rows, heads, text, causal, batch, route):
    n = batch * rows * heads * 128
    q, k, v = (synth(oracle, n, 200 + i) for i in range(3))
    got = run(gpu, qd, q, k, v, batch, rows, rows, heads, text_rows=text, text_causal=causal)
    assert gpu.route() == route
    lim = oracle.t2i_limits(rows, text, causal)
    # one early and the last heads (the split blocks are the last ones)
    for h in {0, heads - 1}:
        c = slice(h * 128, h * 128 + 128)
        for b in range(batch):
            one = [np.ascontiguousarray(x.reshape(batch, rows, -1)[b, :, c]).ravel()
                   for x in (q, k, v)]
            ref = oracle.attention(*one, lim, rows, rows, 1, prescale_rows=text)
            assert rel_l2(oracle.bf16_to_f32(got[b, :, c].copy()),
                          oracle.bf16_to_f32(ref).reshape(rows, 128)) < 5e-3


@pytest.mark.parametrize("q_rows,kv_rows,heads", [(100, 2000, 2), (300, 8192, 1), (4300, 4500, 17)])
def test_split_attention_cached_keys(gpu, qd, oracle, q_rows, kv_rows, heads):
    """Fewer queries than keys (an editing step against cached keys), a table
    of limits with rows that see one key, the first piece's keys, or all."""
    H = heads * 128
    q, k, v = synth(oracle, q_rows * H, 210), synth(oracle, kv_rows * H, 211), synth(oracle, kv_rows * H, 212)
    lim = np.full(q_rows, kv_rows, np.uint32)
    lim[:3] = (1, 64, 65)
    lim[q_rows // 2] = kv_rows // 2
    lim[-1] = 7
    got = run(gpu, qd, q, k, v, 1, q_rows, kv_rows, heads, kv_limit=gpu.put(lim))[0]
    assert "_split_bf16:split=" in gpu.route()
    h = heads - 1
    c = slice(h * 128, h * 128 + 128)
    one = [np.ascontiguousarray(x.reshape(-1, H)[:, c]).ravel() for x in (q, k, v)]
    ref = oracle.bf16_to_f32(oracle.attention(*one, lim, q_rows, kv_rows, 1)).reshape(q_rows, 128)
    f = oracle.bf16_to_f32(got[:, c].copy())
    assert rel_l2(f, ref) < 5e-3
    for r in (0, 1, 2, q_rows // 2, q_rows - 1):
        assert rel_l2(f[r], ref[r]) < 2e-2  # a row of few keys averages no rounding away
    assert np.array_equal(got[0].view(np.uint16), v.reshape(-1, H)[0])  # one key: its V


@pytest.mark.parametrize("q_rows,kv_rows,heads", [(300, 2000, 2), (2100, 2100, 32)])
def test_split_attention_row_alone(gpu, qd, oracle, q_rows, kv_rows, heads):
    """A row's result does not depend on the other rows of its block: the
    same bits where the others have other queries (some a hundred times as
    large, which move their maxima) and other limits."""
    H = heads * 128
    q, k, v = synth(oracle, q_rows * H, 213), synth(oracle, kv_rows * H, 214), synth(oracle, kv_rows * H, 215)
    rng = np.random.default_rng(4)
    lim = rng.integers(1, kv_rows + 1, q_rows).astype(np.uint32)
    lim[5], lim[q_rows - 1] = kv_rows, 70
    keep = np.zeros(q_rows, bool)
    keep[[0, 5, 31, 32, 100, 255, 256, q_rows - 1]] = True
    got = run(gpu, qd, q, k, v, 1, q_rows, kv_rows, heads, kv_limit=gpu.put(lim))[0]
    route = gpu.route()
    assert "_split_bf16:split=" in route
    other = oracle.bf16_to_f32(synth(oracle, q_rows * H, 216)).reshape(q_rows, H)
    other[::3] *= 100.0
    q2 = oracle.f32_to_bf16(np.ascontiguousarray(other, np.float32).ravel()).reshape(q_rows, H)
    q2[keep] = q.reshape(q_rows, H)[keep]
    # the others see few keys each: whole pieces are empty but for the kept rows
    lim2 = np.where(keep, lim, rng.integers(1, 129, q_rows)).astype(np.uint32)
    got2 = run(gpu, qd, q2.ravel(), k, v, 1, q_rows, kv_rows, heads, kv_limit=gpu.put(lim2))[0]
    assert gpu.route() == route
    assert np.array_equal(got[keep], got2[keep])
    assert not np.array_equal(got[~keep], got2[~keep])


def test_split_attention_large_scores(gpu, qd, oracle):
    """Row maxima that differ by hundreds between the pieces: every piece but
    one vanishes, with no overflow."""
    rows, heads = 1024, 1
    q = oracle.f32_to_bf16(np.tile(np.eye(1, 128, dtype=np.float32) * 64, (rows, 1)))
    kf = np.zeros((rows, 128), np.float32)
    kf[:, 0] = np.linspace(-200, 200, rows)
    v = synth(oracle, rows * 128, 221)
    got = run(gpu, qd, q.ravel(), oracle.f32_to_bf16(kf).ravel(), v, 1, rows, rows, heads)[0]
    assert "split=4" in gpu.route()
    lim = np.full(rows, rows, np.uint32)
    ref = oracle.attention(q.ravel(), oracle.f32_to_bf16(kf).ravel(), v, lim, rows, rows, 1)
    assert np.isfinite(oracle.bf16_to_f32(got.ravel())).all()
    assert rel_l2(oracle.bf16_to_f32(got.ravel()), oracle.bf16_to_f32(ref).ravel()) < 5e-3


@pytest.mark.parametrize("causal", [0, 1])
def test_split_attention_more_text_rows_than_keys(gpu, qd, oracle, monkeypatch, causal):
    """Text rows past the last key: the keys that whole blocks count."""
    rows, kv, heads = 2600, 2000, 1
    q, k, v = synth(oracle, rows * 128, 230), synth(oracle, kv * 128, 231), synth(oracle, kv * 128, 232)
    got = run(gpu, qd, q, k, v, 1, rows, kv, heads, text_rows=rows, text_causal=causal)
    assert "split=" in gpu.route()
    monkeypatch.setenv("QW_WORKSPACES", "0")
    whole = qd.Gpu()
    try:
        want = run(whole, qd, q, k, v, 1, rows, kv, heads, text_rows=rows, text_causal=causal)
        assert "split=" not in whole.route()
    finally:
        whole.close()
    a, b = (oracle.bf16_to_f32(x.ravel()).reshape(rows, 128) for x in (got, want))
    for r in (range(0, kv), range(kv, rows)):
        assert rel_l2(a[r], b[r]) < 5e-3
