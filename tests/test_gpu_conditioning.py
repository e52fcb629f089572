"""The conditioning chain in three launches against the separate linears,
activations and reorder, bit for bit: the same sums in the same order, the
same roundings."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,hidden,shift,bias", [
    (1, 256, 0, False), (2, 256, 1, True), (2, 3072, 1, True), (1, 4096, 0, False),
    (2, 1280, 0, True)])  # k-chunks of a lane: a part of one, one, six, eight, two and a half
def test_conditioning_bit_identical(gpu, qd, oracle, rows, hidden, shift, bias):
    H, S, nout, L = hidden, 6 if shift else 4, (1 + shift) * hidden, qd.lib()
    put = lambda n, s, std=0.02: gpu.put(oracle.fill_normal_bf16(n, 31, s, std))  # noqa: E731
    l1, l2 = put(H * 256, 1, 0.1), put(H * H, 2, 0.1)
    mod, out = put(S * H * H, 3, 0.1), put(nout * H, 4)
    b1, b2, bm, bo = (put(n, 5 + i) if bias else None for i, n in enumerate((H, H, S * H, nout)))
    feats = np.random.default_rng(3).uniform(-1, 1, 1 + rows * 256).astype(np.float32)
    base = gpu.put(feats)
    f = base.view(1, rows * 256)  # features at any float
    new = lambda n: gpu.new(n, qd.BF16)  # noqa: E731
    got = [new(rows * H), new(rows * S * H), new(rows * nout)]
    h = lambda t: t.h if t is not None else None  # noqa: E731
    d = qd.ConditioningDesc(f.h, l1.h, h(b1), l2.h, h(b2), mod.h, h(bm), out.h, h(bo),
                            new(rows * H).h, new(rows * H).h, *(t.h for t in got), rows, H, shift)
    wide, silu = new(rows * H), new(rows * H)
    d.wide, d.silu = wide.h, silu.h
    gpu.check(L.qw_gpu_conditioning_bf16(gpu.h, C.byref(d)), "conditioning")
    fb, w, sl, t, raw, mo, no = (new(n) for n in (rows * 256, rows * H, rows * H, rows * H,
                                                  rows * S * H, rows * S * H, rows * nout))
    gpu.check(L.h3_gpu_cast_f32_to_bf16(gpu.h, fb.h, f.h, rows * 256), "cast")
    gpu.linear(w, fb, l1, rows, 256, H, bias=b1)
    gpu.check(L.h3_gpu_silu_bf16(gpu.h, w.h, w.h, rows * H), "silu")
    gpu.linear(t, w, l2, rows, H, H, bias=b2)
    gpu.check(L.h3_gpu_silu_bf16(gpu.h, sl.h, t.h, rows * H), "silu")
    gpu.linear(no, sl, out, rows, H, nout, bias=bo)
    gpu.linear(raw, sl, mod, rows, H, S * H, bias=bm)
    gpu.check(L.qw_gpu_modulation_reorder_bf16(gpu.h, mo.h, raw.h, rows, H, shift), "reorder")
    gpu.submit()
    for a, b in zip(got, (t, mo, no)):
        assert np.array_equal(a.read(), b.read())


def test_conditioning_refusals(gpu, qd):
    H, rows, L = 256, 1, qd.lib()
    t = [gpu.new(n, ty) for n, ty in [(256, qd.F32), (H * 256, qd.BF16), (H * H, qd.BF16),
                                      (4 * H * H, qd.BF16), (H * H, qd.BF16)]]
    o = [gpu.new(n, qd.BF16) for n in (H, H, H, 4 * H, H)]
    ok = lambda **kw: L.qw_gpu_conditioning_bf16(gpu.h, C.byref(qd.ConditioningDesc(  # noqa: E731
        kw.get("features", t[0]).h, t[1].h, None, t[2].h, None, t[3].h, None, t[4].h, None,
        *(x.h for x in o), kw.get("rows", rows), kw.get("hidden", H), kw.get("shift", 0))))
    assert ok()
    assert not ok(rows=0) and not ok(rows=3) and not ok(rows=2)
    assert not ok(features=o[0])  # bf16
    assert not ok(shift=1)  # six slots do not fit
    assert not ok(hidden=257) and not ok(hidden=512)
    gpu.submit()


def test_conditioning_overlaps(gpu, qd, oracle):
    """A stage whose output lies over its input, or silu over temb, is
    refused; the modulation over the final norm's factor leaves what separate
    linears do: the modulation whole, after the factor."""
    H, rows, L = 256, 2, qd.lib()
    put = lambda n, s: gpu.put(oracle.fill_normal_bf16(n, 31, s, 0.1))  # noqa: E731
    f = gpu.put(np.random.default_rng(3).uniform(-1, 1, rows * 256).astype(np.float32))
    w = [put(n, i) for i, n in enumerate((H * 256, H * H, 4 * H * H, H * H))]
    names = ("wide", "silu", "temb", "modulation", "norm_out")
    size = dict(zip(names, (rows * H, rows * H, rows * H, 4 * rows * H, rows * H)))

    def call(**views):
        o = {n: views.get(n) or gpu.new(size[n], qd.BF16) for n in names}
        d = qd.ConditioningDesc(f.h, w[0].h, None, w[1].h, None, w[2].h, None, w[3].h, None,
                                *(o[n].h for n in names), rows, H, 0)
        ok = L.qw_gpu_conditioning_bf16(gpu.h, C.byref(d))
        gpu.submit()
        return {n: t.read() for n, t in o.items()} if ok else None

    ref = call()
    buf = gpu.new(8 * rows * H, qd.BF16)
    for a, b in (("wide", "temb"), ("wide", "silu"), ("temb", "silu"), ("silu", "modulation"),
                 ("silu", "norm_out")):
        for off in (0, size[a] - 8):
            assert call(**{a: buf.view(0, size[a]), b: buf.view(off, size[b])}) is None
        assert call(**{a: buf.view(0, size[a]), b: buf.view(size[a], size[b])}) is not None
    for off in (0, 3 * rows * H + 8):
        got = call(modulation=buf.view(0, size["modulation"]), norm_out=buf.view(off, size["norm_out"]))
        assert np.array_equal(got["modulation"], ref["modulation"])
        assert np.array_equal(got["temb"], ref["temb"])
        tail = max(0, off + size["norm_out"] - size["modulation"])
        if tail:
            assert np.array_equal(got["norm_out"][-tail:], ref["norm_out"][-tail:])
