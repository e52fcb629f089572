"""The work that a user of this library has it do, as cases that can be timed
and checked: the DiT denoising forward and its parts, each through a public
entry point of include/*.h (by way of qdit.py, the ctypes binding).

Sizes are those of the two geometries that qwen_dit.h names (the benchmark
geometry, "baseline": hidden 3072, 24 heads, GELU MLP, shift, biases; and
"reference": hidden 4096, 32 heads, SwiGLU, no biases), at images of 256^2 to
1024^2 (16 x 16 to 64 x 64 tokens) with some tens to hundreds of text rows.

A case is one call of one kind:
  conditioning  qw_dit_conditioning: timestep features -> modulation
  norm          qw_gpu_layer_norm_mod_shift_bf16 over a hidden state
  linear        qw_gpu_linear with the epilogue the block gives that layer
  attention     qw_gpu_attention_bf16
  block         qw_dit_block
  forward       qw_dit_forward_batch, all its layers
  ti2i          qw_dit_forward_ti2i, a sampling step on cached K/V
"""
import ctypes as C
import importlib.util
import math
import os

import numpy as np
import torch

_ROOT = os.getcwd()
_spec = importlib.util.spec_from_file_location(
    "qdit", os.path.join(_ROOT, "qwen-metal_amd", "qdit.py"))
qd = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(qd)

# the two geometries of qwen_dit.h (qw_dit_config_baseline / _reference)
GEOMETRY = {
    "baseline": dict(hidden=3072, heads=24, mlp_width=12288, text_dim=4096, z_dim=64,
                     mlp_act=qd.MLP_GELU_TANH, adaln_shift=1, has_bias=1, text_causal=0),
    "reference": dict(hidden=4096, heads=32, mlp_width=12288, text_dim=4096, z_dim=64,
                      mlp_act=qd.MLP_SWIGLU, adaln_shift=0, has_bias=0, text_causal=1),
}
EPS = 1e-6
SCALE = 1.0 / math.sqrt(128.0)


def listed():
    return [
        # once per denoising step: the smallest call, a chain of launches on two rows
        dict(name="conditioning", kind="conditioning", geometry="baseline", mod_rows=2),
        # a prompt's embedding into the joint sequence: few and ragged rows
        dict(name="linear_text_100", kind="linear", geometry="baseline", layer="text", rows=100,
             text_rows=100, int8=False),
        # twice per block of a 1024^2 step with guidance (two stacked branches)
        dict(name="norm_8704", kind="norm", geometry="baseline", rows=8704, text_rows=256),
        # one linear of the bf16 sweep at 1024^2 without guidance
        dict(name="linear_up_4352", kind="linear", geometry="baseline", layer="up", rows=4352,
             text_rows=256, int8=False),
        # the largest int8 linear of the 1024^2 step with guidance
        dict(name="linear_down_8704_int8", kind="linear", geometry="baseline", layer="down",
             rows=8704, text_rows=256, int8=True),
        # attention of the 512^2 step, and of the 1024^2 step with guidance
        dict(name="attention_1152", kind="attention", heads=24, batch=1, text_rows=128,
             image_rows=1024, cached_rows=0, causal=False),
        dict(name="attention_2x4352", kind="attention", heads=24, batch=2, text_rows=256,
             image_rows=4096, cached_rows=0, causal=False),
        # one block of a 256^2, a 512^2 and a 1024^2 image; the last in the
        # reference geometry with a short prompt, so a ragged row count
        dict(name="block_320", kind="block", geometry="baseline", int8=False, text_rows=64, gh=16,
             gw=16),
        dict(name="block_1152", kind="block", geometry="baseline", int8=False, text_rows=128,
             gh=32, gw=32),
        dict(name="block_4119_reference", kind="block", geometry="reference", int8=False,
             text_rows=23, gh=64, gw=64),
        # editing: the second and later sampling steps, against the condition
        # image's cached K/V (a few layers of the model)
        dict(name="ti2i_4096_of_8512", kind="ti2i", geometry="reference", int8=False, layers=4,
             text_rows=256, cond_gh=64, cond_gw=64, text_rows2=64, gh=64, gw=64),
        # the whole model: one 1024^2 step with guidance, int8 weights
        dict(name="forward_1024_cfg_int8", kind="forward", geometry="baseline", int8=True,
             batch=2, text_rows=256, gh=64, gw=64, layers=32),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["conditioning", "norm", "linear", "linear", "attention", "attention",
                       "block", "block", "forward", "ti2i"])
    geometry = rng.choice(["baseline", "reference"])
    text = _log_int(rng, 9, 384)
    gh, gw = rng.randint(14, 64), rng.randint(14, 64)
    int8 = rng.random() < 0.4
    if kind == "conditioning":
        return dict(kind=kind, geometry=geometry, mod_rows=rng.choice([1, 2]),
                    sigma_ppm=rng.randint(1, 999999))
    if kind == "norm":
        rows = _log_int(rng, 64, 8704)
        return dict(kind=kind, geometry=geometry, rows=rows, text_rows=min(rows, text))
    if kind == "linear":
        rows = _log_int(rng, 9, 8704)
        layer = rng.choice(["qkv", "out", "up", "down", "text"])
        return dict(kind=kind, geometry=geometry, layer=layer, rows=rows,
                    text_rows=min(rows, text), int8=int8 and layer != "text")
    if kind == "attention":
        heads = GEOMETRY[geometry]["heads"]
        cached = rng.choice([0, 0, rng.randint(100, 4500)])
        return dict(kind=kind, heads=heads, batch=1 if cached else rng.choice([1, 2]),
                    text_rows=0 if cached else text, image_rows=gh * gw, cached_rows=cached,
                    causal=geometry == "reference")
    if kind == "block":
        return dict(kind=kind, geometry=geometry, int8=int8, text_rows=text, gh=gh, gw=gw)
    if kind == "forward":
        return dict(kind=kind, geometry=geometry, int8=int8, batch=rng.choice([1, 2]),
                    text_rows=text, gh=gh, gw=gw, layers=rng.randint(1, 4))
    return dict(kind="ti2i", geometry=geometry, int8=int8, layers=rng.randint(1, 3),
                text_rows=text, cond_gh=rng.randint(14, 48), cond_gw=rng.randint(14, 48),
                text_rows2=_log_int(rng, 9, 96), gh=gh, gw=gw)


# ---- device tensors -------------------------------------------------------

_gpu = None


def _context():
    """One context per program, as a user's program has."""
    global _gpu
    if _gpu is None:
        torch.cuda.init()
        _gpu = qd.Gpu()
    return _gpu


class _Memory:
    def __init__(self, ptr, n, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (ptr, False),
                                         "version": 2}


_TYPES = {qd.F32: ("<f4", None), qd.BF16: ("<i2", torch.bfloat16), qd.I8: ("|i1", None),
          qd.U32: ("<i4", None)}


def _torch(handle, n, dtype, owner):
    """A torch view of a library tensor's memory; keeps `owner` alive."""
    typestr, as_type = _TYPES[dtype]
    t = torch.as_tensor(_Memory(qd.lib().h3_gpu_tensor_device_ptr(handle), n, typestr, owner),
                        device="cuda")
    return t.view(as_type) if as_type is not None else t


def _view(t, *shape):
    return _torch(t.h, t.n, t.dtype, t).view(*shape)


def _normal(gen, n, std=1.0, mean=0.0):
    """A library tensor of n bf16 values N(mean, std)."""
    t = _context().new(n, qd.BF16)
    v = _view(t, n)
    step = 1 << 26
    for i in range(0, n, step):
        m = min(step, n - i)
        v[i:i + m] = torch.randn(m, generator=gen, device="cuda") * std + mean
    return t


def _put(a):
    a = np.ascontiguousarray(a)
    t = _context().new(a.size, {"float32": qd.F32, "uint32": qd.U32}[str(a.dtype)])
    t.write(a)
    return t


def _rope(text_rows, gh, gw):
    """The t2i tables, f32 [text + gh gw, 64] each."""
    cos = np.empty((text_rows + gh * gw, 64), np.float32)
    sin = np.empty_like(cos)
    qd.lib().qw_pipe_rope_tables_host(text_rows, gh, gw, cos.ctypes.data, sin.ctypes.data)
    return cos, sin


def _row_map(rows, text_rows, batch=1):
    """Text rows ride modulation row 1 (t = 0), image rows row 0."""
    return np.tile((np.arange(rows) < text_rows).astype(np.uint32), batch)


def _slots(geo):
    return 6 if geo["adaln_shift"] else 4


def _layer_shape(geo, layer):
    """(k, cols) of a linear."""
    H, F = geo["hidden"], geo["mlp_width"]
    up = 2 * F if geo["mlp_act"] == qd.MLP_SWIGLU else F
    return {"qkv": (H, 3 * H), "out": (H, H), "up": (H, up), "down": (F, H),
            "text": (geo["text_dim"], H)}[layer]


class _Segment(C.Structure):
    _fields_ = [("rows", C.c_uint32), ("is_image", C.c_int), ("src_offset", C.c_uint32)]


class _State:
    """The inputs, weights and outputs of a case, by attribute."""

    def __init__(self, **kw):
        self.__dict__.update(kw)

    def __del__(self):
        dit = self.__dict__.pop("dit", None)
        if dit is not None:
            dit.close()


def _model(case, seed, layers):
    geo = GEOMETRY[case["geometry"]]
    return qd.Dit(_context(), dict(geo, layers=layers, int8_weights=int(case.get("int8", False))),
                  seed)


def prepare(case, seed):
    gpu = _context()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind = case["kind"]
    geo = GEOMETRY.get(case.get("geometry"))
    H = geo["hidden"] if geo else 0
    s = _State(case=dict(case), gpu=gpu)
    if kind == "conditioning":
        n = case["mod_rows"]
        # sigma of the step (row 0); conditioning rows ride t = 0 (row 1)
        sigma = case.get("sigma_ppm", 1 + (seed * 7919) % 999999) / 1e6
        feats = np.empty((n, 256), np.float32)
        sig = np.array([sigma, 0.0][:n], np.float32)
        qd.lib().qw_dit_timestep_features(sig.ctypes.data, n, feats.ctypes.data)
        s.dit, s.features, s.mod_rows = _model(case, seed, 1), _put(feats), n
        nout = (2 if geo["adaln_shift"] else 1) * H
        s.temb, s.modulation, s.norm_out = (gpu.new(n * H, qd.BF16),
                                            gpu.new(n * _slots(geo) * H, qd.BF16),
                                            gpu.new(n * nout, qd.BF16))
        s.result = [_view(s.temb, n, H), _view(s.modulation, n, -1), _view(s.norm_out, n, nout)]
    elif kind == "norm":
        n = case["rows"]
        s.x, s.out = _normal(gen, n * H), gpu.new(n * H, qd.BF16)
        s.modulation = _normal(gen, 2 * _slots(geo) * H, 0.2)
        s.row_map = _put(_row_map(n, case["text_rows"]))
        s.args = (gpu.h, s.out.h, s.x.h, s.modulation.h, s.row_map.h, n, H, _slots(geo), 0,
                  4 if geo["adaln_shift"] else -1, EPS)
        s.result = _view(s.out, n, H)
    elif kind == "linear":
        n, layer = case["rows"], case["layer"]
        k, cols = _layer_shape(geo, layer)
        s.x, s.weight, s.wscale = _normal(gen, n * k), _normal(gen, cols * k, 0.02), None
        if case["int8"]:
            s.wide, s.weight, s.wscale = s.weight, gpu.new(cols * k, qd.I8), gpu.new(cols, qd.F32)
            torch.cuda.synchronize()
            gpu.check(qd.lib().h3_gpu_quantize_weight_int8(gpu.h, s.weight.h, s.wscale.h, s.wide.h,
                                                           cols, k), "quantize")
            gpu.submit()
            s.wide = None
        s.bias = _normal(gen, cols, 0.02) if geo["has_bias"] else None
        s.kw = dict(bias=s.bias, wscale=s.wscale)
        s.out = gpu.new(n * cols, qd.BF16)
        if layer in ("out", "down"):  # gated into the residual, in place
            s.out = _normal(gen, n * cols)
            s.modulation = _normal(gen, 2 * _slots(geo) * cols, 0.2)
            s.row_map = _put(_row_map(n, case["text_rows"]))
            s.kw.update(epilogue=qd.LINEAR_GATE, modulation=s.modulation, row_map=s.row_map,
                        slots=_slots(geo), gate_slot=2 if layer == "out" else 3)
        elif layer == "qkv":
            s.norm_q, s.norm_k = _normal(gen, 128, 0.02, 1.0), _normal(gen, 128, 0.02, 1.0)
            s.cos, s.sin = (_put(t) for t in _rope(case["text_rows"], 1, max(1, n - case["text_rows"])))
            s.kw.update(epilogue=qd.LINEAR_QKNORM,
                        qknorm=(s.norm_q, s.norm_k, s.cos, s.sin, s.cos.n // 64, EPS))
        elif layer == "text" or geo["mlp_act"] == qd.MLP_GELU_TANH:
            s.kw.update(epilogue=qd.LINEAR_GELU)
        s.args = (s.out, s.x, s.weight, n, k, cols)
        s.result = _view(s.out, n, cols)
    elif kind == "attention":
        B, heads, T = case["batch"], case["heads"], case["text_rows"]
        H, R = heads * 128, T + case["image_rows"]
        if case["cached_rows"]:  # queries of the target against cached keys
            kv = R + case["cached_rows"]
            s.q, s.k, s.v = (_normal(gen, n * H) for n in (R * 3, kv, kv))
            s.args = (s.q, s.k, s.v, 1, R, kv, heads, 3 * H, H, H, H)
            s.kw = {}
        else:  # the fused q | k | v projection
            s.q = _normal(gen, B * R * 3 * H)
            s.args = (s.q, s.q, s.q, B, R, R, heads, 3 * H, 3 * H, 3 * H, H)
            s.kw = dict(k_offset=H, v_offset=2 * H, text_rows=T, text_causal=int(case["causal"]))
        qk = _view(s.q, B * R, 3, heads, 128)  # q and k come RMS-normalised per head
        for t in ((qk[:, 0],) if case["cached_rows"] else (qk[:, 0], qk[:, 1])):
            f = t.float()
            t.copy_(f / f.square().mean(-1, keepdim=True).sqrt())
        if case["cached_rows"]:
            t = _view(s.k, -1, heads, 128)
            f = t.float()
            t.copy_(f / f.square().mean(-1, keepdim=True).sqrt())
        s.out = gpu.new(B * R * H, qd.BF16)
        s.result = _view(s.out, B * R, H)
    elif kind == "block":
        T, R = case["text_rows"], case["text_rows"] + case["gh"] * case["gw"]
        s.dit = _model(case, seed, 1)
        s.hidden, s.modulation = _normal(gen, R * H), _normal(gen, 2 * _slots(geo) * H, 0.2)
        s.cos, s.sin = (_put(t) for t in _rope(T, case["gh"], case["gw"]))
        s.row_map = _put(_row_map(R, T))
        s.args = (0, s.hidden, s.modulation, s.cos, s.sin, s.row_map, R, T)
        s.result = _view(s.hidden, R, H)  # updated in place
    elif kind == "forward":
        B, T, I = case["batch"], case["text_rows"], case["gh"] * case["gw"]
        s.dit = _model(case, seed, case["layers"])
        s.text = _normal(gen, B * T * geo["text_dim"])
        # both branches of guidance denoise the same latents
        one = torch.randn(I * geo["z_dim"], generator=gen, device="cuda").to(torch.bfloat16)
        s.latents = gpu.new(B * I * geo["z_dim"], qd.BF16)
        _view(s.latents, B, -1).copy_(one.expand(B, -1))
        s.cos, s.sin = (_put(t) for t in _rope(T, case["gh"], case["gw"]))
        s.out = gpu.new(B * (T + I) * geo["z_dim"], qd.BF16)
        s.sigma = _sigma(seed)
        s.args = (s.text, T, s.latents, I, B, s.sigma, s.cos, s.sin, s.out)
        s.result = _view(s.out, B, T + I, geo["z_dim"])
    else:
        runs = _ti2i_runs(case)
        rows, target = sum(r[0] for r in runs), runs[-1][0]
        s.dit = _model(case, seed, case["layers"])
        s.text = _normal(gen, (case["text_rows"] + case["text_rows2"]) * geo["text_dim"])
        s.latents = _normal(gen, (runs[1][0] + target) * geo["z_dim"])
        s.segs = (_Segment * len(runs))(*(_Segment(*r) for r in runs))
        s.cos, s.sin = (_put(t) for t in _ti2i_rope(case))
        s.out = gpu.new(rows * geo["z_dim"], qd.BF16)
        s.err = C.create_string_buffer(1024)
        s.sigma = _sigma(seed)
        torch.cuda.synchronize()
        _ti2i(s, 1.0)  # the first step: a full pass that fills the cache
        # a cached step writes the target's rows
        s.result = _view(s.out, rows, geo["z_dim"])[rows - target:]
    torch.cuda.synchronize()
    return s


def _sigma(seed):
    return (100 + (seed * 7919) % 800) / 1000.0


def _ti2i_runs(case):
    """(rows, is_image, source row): text, condition image, text, target."""
    c, t = case["cond_gh"] * case["cond_gw"], case["gh"] * case["gw"]
    return [(case["text_rows"], 0, 0), (c, 1, 0), (case["text_rows2"], 0, case["text_rows"]),
            (t, 1, c)]


def _ti2i_rope(case):
    h = np.array([case["cond_gh"], case["gh"]], np.uint32)
    w = np.array([case["cond_gw"], case["gw"]], np.uint32)
    t = np.array([case["text_rows"], case["text_rows2"]], np.uint32)
    fill = qd.lib().qw_pipe_rope_tables_blocks_host
    n = fill(h.ctypes.data, w.ctypes.data, t.ctypes.data, 2, None, None)
    cos, sin = np.empty((n, 64), np.float32), np.empty((n, 64), np.float32)
    fill(h.ctypes.data, w.ctypes.data, t.ctypes.data, 2, cos.ctypes.data, sin.ctypes.data)
    return cos, sin


def _ti2i(s, sigma):
    if not qd.lib().qw_dit_forward_ti2i(s.dit.h, s.text.h, s.latents.h, s.segs, len(s.segs), 0,
                                        s.cos.h, s.sin.h, sigma, s.out.h, s.err, 1024):
        raise RuntimeError(s.err.value.decode())


def run(s):
    kind = s.case["kind"]
    if kind == "conditioning":
        err = C.create_string_buffer(256)
        if not qd.lib().qw_dit_conditioning(s.dit.h, s.features.h, s.mod_rows, s.temb.h,
                                            s.modulation.h, s.norm_out.h, err, 256):
            raise RuntimeError(err.value.decode())
    elif kind == "norm":
        s.gpu.check(qd.lib().qw_gpu_layer_norm_mod_shift_bf16(*s.args), "norm")
    elif kind == "linear":
        s.gpu.linear(*s.args, **s.kw)
    elif kind == "attention":
        s.gpu.attention(s.out, *s.args, **s.kw)
    elif kind == "block":
        s.dit.block(*s.args)
    elif kind == "forward":
        s.dit.forward_batch(*s.args)
    else:
        _ti2i(s, s.sigma)
    return s.result


# ---- work -----------------------------------------------------------------


def _pairs(batch, text_rows, image_rows, cached_rows, causal):
    """Visible (query, key) pairs."""
    R = text_rows + image_rows
    text = text_rows * (text_rows + 1) // 2 if causal else text_rows * text_rows
    return batch * (text + image_rows * (R + cached_rows))


def _block_work(geo, int8, rows, pairs, cached_rows=0):
    """(bytes, flops) of one block's weights, hidden state and products."""
    H, F = geo["hidden"], geo["mlp_width"]
    w = sum(k * n for k, n in (_layer_shape(geo, x) for x in ("qkv", "out", "up", "down")))
    return (w * (1 if int8 else 2) + 2 * rows * H * 2 + 2 * cached_rows * H * 2,
            2 * rows * w + 4 * H * pairs)


def _conditioning_bytes(geo):
    H = geo["hidden"]
    return 2 * H * (256 + H + (_slots(geo) + 1 + geo["adaln_shift"]) * H)


def _embed_work(geo, text_rows, image_rows):
    H, D, Z = geo["hidden"], geo["text_dim"], geo["z_dim"]
    w = (D * H + H * H) if text_rows else 0
    return (2 * (w + Z * H + text_rows * D + image_rows * Z),
            2 * (text_rows * w + image_rows * Z * H))


def work(case):
    kind = case["kind"]
    geo = GEOMETRY.get(case.get("geometry"))
    H = geo["hidden"] if geo else 0
    if kind == "conditioning":
        b = _conditioning_bytes(geo)
        return {"bytes": b, "flops": b * case["mod_rows"]}
    if kind == "norm":
        return {"bytes": 4 * case["rows"] * H + 4 * case["rows"], "flops": 9 * case["rows"] * H}
    if kind == "linear":
        n = case["rows"]
        k, cols = _layer_shape(geo, case["layer"])
        gated = case["layer"] in ("out", "down")
        return {"bytes": k * cols * (1 if case["int8"] else 2) + 2 * n * k +
                (4 if gated else 2) * n * cols,
                "flops": 2 * n * k * cols}
    if kind == "attention":
        H, R = case["heads"] * 128, case["text_rows"] + case["image_rows"]
        p = _pairs(case["batch"], case["text_rows"], case["image_rows"], case["cached_rows"],
                   case["causal"])
        return {"bytes": 2 * H * case["batch"] * (4 * R + 2 * case["cached_rows"]),
                "flops": 4 * H * p}
    T, I = case["text_rows"], case["gh"] * case["gw"]
    if kind == "block":
        b, f = _block_work(geo, case["int8"], T + I, _pairs(1, T, I, 0, geo["text_causal"]))
        return {"bytes": b, "flops": f}
    if kind == "forward":
        B = case["batch"]
        M = B * (T + I)
        b, f = _block_work(geo, case["int8"], M, _pairs(B, T, I, 0, geo["text_causal"]))
        eb, ef = _embed_work(geo, B * T, B * I)
    else:
        B, M = 1, I
        cached = T + case["text_rows2"] + case["cond_gh"] * case["cond_gw"]
        b, f = _block_work(geo, case["int8"], M, _pairs(1, 0, I, cached, 0), cached)
        eb, ef = _embed_work(geo, 0, I)
    # between blocks the hidden state need not leave the chip's caches: its
    # reads and writes count once, the weights in every layer
    b -= 4 * M * H
    return {"bytes": case["layers"] * b + 4 * M * H + eb + _conditioning_bytes(geo) +
            4 * M * geo["z_dim"],
            "flops": case["layers"] * f + ef + 2 * M * H * geo["z_dim"]}


def tolerance(case):
    """Outputs and the operands between kernels are bf16 (8 bits: 2^-9 = 2e-3
    relative per rounding), sums fp32. Each bound is about four times what the
    kind measures against 64 bits."""
    kind = case["kind"]
    if kind in ("forward", "ti2i"):
        # random weights: each layer amplifies the roundings of those before it
        return {"rel": 0.03, "max": 0.9}
    return {"rel": {"conditioning": 1.6e-2, "norm": 7e-3, "linear": 1e-2, "attention": 1e-2,
                    "block": 1.2e-2}[kind]}


# ---- the same in 64 bits, in plain torch ----------------------------------


def _d(t):
    """A library tensor's values in 64 bits."""
    return _view(t, t.n).double()


def _fill(n, seed, stream, std=0.02, offset=0.0):
    """A weight of the model by its documented generator stream."""
    gpu = _context()
    t = gpu.new(n, qd.BF16)
    gpu.check(qd.lib().qw_gpu_fill_normal_bf16(gpu.h, t.h, 0, n, seed, stream, std, offset), "fill")
    gpu.submit()
    return _d(t)


# weight streams of qw_dit_create_random (qwen_dit.h: QW_W_*, QW_L_*)
_W = {n: i + 1 for i, n in enumerate(
    ["img_in", "img_in_b", "txt_norm", "txt_in1", "txt_in1_b", "txt_in2", "txt_in2_b", "time_l1",
     "time_l1_b", "time_l2", "time_l2_b", "mod", "mod_b", "norm_out", "norm_out_b", "proj_out",
     "proj_out_b"])}
_L = {n: i + 1 for i, n in enumerate(
    ["qkv", "qkv_b", "out", "out_b", "up", "up_b", "down", "down_b", "norm_q", "norm_k"])}


def _apply(geo, seed, name, n, k, x):
    y = x @ _fill(n * k, seed, _W[name]).view(n, k).T
    return y + _fill(n, seed, _W[name + "_b"]) if geo["has_bias"] else y


def _silu(x):
    return x * torch.sigmoid(x)


def _gelu(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _features(sigmas):
    t = torch.tensor(sigmas, dtype=torch.float64, device="cuda")[:, None] * 1000.0
    i = torch.arange(128, dtype=torch.float64, device="cuda")
    a = t * 10000.0 ** (-i / 128.0)
    return torch.cat([a.cos(), a.sin()], 1)


def _conditioning64(geo, seed, features):
    """temb, modulation slots [rows, S, H], norm_out [rows, 1 or 2, H]"""
    H, S, sh = geo["hidden"], _slots(geo), geo["adaln_shift"]
    temb = _apply(geo, seed, "time_l2", H, H, _silu(_apply(geo, seed, "time_l1", H, 256, features)))
    raw = _apply(geo, seed, "mod", S * H, H, _silu(temb)).view(-1, S, H)
    out = _apply(geo, seed, "norm_out", (1 + sh) * H, H, _silu(temb))
    if sh:  # shift, scale, gate of either half
        order = [raw[:, 1], raw[:, 4], raw[:, 2].tanh(), raw[:, 5].tanh(), raw[:, 0], raw[:, 3]]
    else:
        order = [raw[:, 0], raw[:, 2], raw[:, 1].tanh(), raw[:, 3].tanh()]
    return temb, torch.stack(order, 1), out.view(-1, 1 + sh, H)


def _norm64(x, scale, shift=None):
    x = x - x.mean(-1, keepdim=True)
    y = x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * (1.0 + scale)
    return y if shift is None else y + shift


def _qk64(x, w, cos, sin):
    """Per-head RMS norm and rotation of [rows, heads, 128]."""
    x = x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w
    a, b, c, s = x[..., 0::2], x[..., 1::2], cos[:, None], sin[:, None]
    return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)


def _attend64(q, k, v, limit):
    """[rows, heads, 128] queries, each against its first limit[row] keys."""
    out = torch.empty_like(q)
    key = torch.arange(k.shape[0], device="cuda")
    for h in range(q.shape[1]):
        kh, vh = k[:, h].contiguous().T.contiguous(), v[:, h].contiguous()
        for r in range(0, q.shape[0], 2048):
            s = (q[r:r + 2048, h].contiguous() @ kh) * SCALE
            s.masked_fill_(key[None] >= limit[r:r + 2048, None], -math.inf)
            out[r:r + 2048, h] = torch.softmax(s, -1) @ vh
    return out


def _limits(text_rows, rows, causal):
    r = torch.arange(rows, device="cuda")
    text = r + 1 if causal else torch.full_like(r, text_rows)
    return torch.where(r < text_rows, text, torch.full_like(r, rows))


def _weights64(dit, geo, seed, layer):
    H, F = geo["hidden"], geo["mlp_width"]
    fields = {"qkv": (0, 1, 2), "out": (3,), "up": (4,), "down": (5,)}
    w = {}
    for name, ids in fields.items():
        k, n = _layer_shape(geo, name)
        parts = []
        for f in ids:
            h, rows = dit.block_tensor(layer, f), n // len(ids)
            t = _torch(h, rows * k, qd.lib().h3_gpu_tensor_dtype(h), dit).double().view(rows, k)
            sc = qd.lib().qw_dit_block_scales(dit.h, layer, f)
            parts.append(t * _torch(sc, rows, qd.F32, dit).double()[:, None] if sc else t)
        w[name] = torch.cat(parts).T
        at = 256 * (layer + 1)
        w[name + "_b"] = _fill(n, seed, at + _L[name + "_b"]) if geo["has_bias"] else 0.0
    w["norm_q"], w["norm_k"] = (_fill(128, seed, at + _L[x], 0.02, 1.0)
                                for x in ("norm_q", "norm_k"))
    return w


def _block64(geo, w, hidden, mod, row_map, cos, sin, limit, batch=1):
    """hidden [batch rows, H], mod [rows, slots, H]"""
    H, sh = geo["hidden"], geo["adaln_shift"]
    R = hidden.shape[0] // batch
    m = [mod[:, i][row_map] for i in range(_slots(geo))] + [None, None]
    x = _norm64(hidden, m[0], m[4] if sh else None)
    qkv = (x @ w["qkv"] + w["qkv_b"]).view(batch, R, 3, geo["heads"], 128)
    att = torch.cat([_attend64(_qk64(b[:, 0], w["norm_q"], cos, sin),
                               _qk64(b[:, 1], w["norm_k"], cos, sin), b[:, 2], limit)
                     for b in qkv]).flatten(1)
    hidden = hidden + (att @ w["out"] + w["out_b"]) * m[2]
    x = _norm64(hidden, m[1], m[5] if sh else None) @ w["up"] + w["up_b"]
    if geo["mlp_act"] == qd.MLP_SWIGLU:
        x = _silu(x[:, :geo["mlp_width"]]) * x[:, geo["mlp_width"]:]
    else:
        x = _gelu(x)
    return hidden + (x @ w["down"] + w["down_b"]) * m[3]


def _text64(geo, seed, text):
    H, D = geo["hidden"], geo["text_dim"]
    x = text / (text.square().mean(-1, keepdim=True) + EPS).sqrt()
    x = x * (_fill(D, seed, _W["txt_norm"]) + 1.0)
    return _apply(geo, seed, "txt_in2", H, H, _gelu(_apply(geo, seed, "txt_in1", H, D, x)))


def _final64(geo, seed, hidden, norm_out, row_map):
    sh = norm_out[:, 1][row_map] if geo["adaln_shift"] else None
    x = _norm64(hidden, norm_out[:, 0][row_map], sh)
    return _apply(geo, seed, "proj_out", geo["z_dim"], geo["hidden"], x)


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    geo = GEOMETRY.get(case.get("geometry"))
    H = geo["hidden"] if geo else 0
    if kind == "conditioning":
        temb, mod, out = _conditioning64(geo, seed, _d(s.features).view(-1, 256))
        return [temb, mod.flatten(1), out.flatten(1)]
    if kind in ("norm", "block"):
        mod = _d(s.modulation).view(2, -1, H)
        rm = _view(s.row_map, -1).long()
    if kind == "norm":
        return _norm64(_d(s.x).view(-1, H), mod[:, 0][rm], mod[:, 4][rm] if geo["adaln_shift"] else None)
    if kind == "linear":
        k, cols = _layer_shape(geo, case["layer"])
        w = _d(s.weight).view(cols, k)
        if s.wscale is not None:
            w = w * _d(s.wscale)[:, None]
        y = _d(s.x).view(-1, k) @ w.T
        if s.bias is not None:
            y = y + _d(s.bias)
        epi = s.kw.get("epilogue", qd.LINEAR_STORE)
        if epi == qd.LINEAR_GELU:
            y = _gelu(y)
        elif epi == qd.LINEAR_GATE:
            gate = _d(s.modulation).view(2, -1, cols)[:, s.kw["gate_slot"]]
            y = _d(s.out).view(-1, cols) + y * gate[_view(s.row_map, -1).long()]
        elif epi == qd.LINEAR_QKNORM:
            y = y.view(y.shape[0], 3, -1, 128)
            cos, sin = (_d(t).view(-1, 64)[:y.shape[0]] for t in (s.cos, s.sin))
            y = torch.stack([_qk64(y[:, 0], _d(s.norm_q), cos, sin),
                             _qk64(y[:, 1], _d(s.norm_k), cos, sin), y[:, 2]], 1).flatten(1)
        return y
    if kind == "attention":
        heads, T = case["heads"], case["text_rows"]
        R = T + case["image_rows"]
        q = _d(s.q).view(case["batch"], R, 3, heads, 128)
        if case["cached_rows"]:
            k, v = (_d(t).view(-1, heads, 128) for t in (s.k, s.v))
            limit = torch.full((R,), k.shape[0], device="cuda")
            return _attend64(q[0, :, 0], k, v, limit).flatten(1)
        limit = _limits(T, R, case["causal"])
        return torch.cat([_attend64(b[:, 0], b[:, 1], b[:, 2], limit) for b in q]).flatten(1)
    if kind == "block":
        T, R = case["text_rows"], case["text_rows"] + case["gh"] * case["gw"]
        return _block64(geo, _weights64(s.dit, geo, seed, 0), _d(s.hidden).view(R, H), mod, rm,
                        _d(s.cos).view(-1, 64), _d(s.sin).view(-1, 64),
                        _limits(T, R, geo["text_causal"]))
    cos, sin = _d(s.cos).view(-1, 64), _d(s.sin).view(-1, 64)
    _, mod, norm_out = _conditioning64(geo, seed, _features([s.sigma, 0.0]))
    text, lat = _d(s.text).view(-1, geo["text_dim"]), _d(s.latents).view(-1, geo["z_dim"])
    img = _apply(geo, seed, "img_in", H, geo["z_dim"], lat)
    txt = _text64(geo, seed, text)
    if kind == "forward":
        B, T, I = case["batch"], case["text_rows"], case["gh"] * case["gw"]
        hidden = torch.cat([x for b in range(B) for x in (txt[b * T:(b + 1) * T],
                                                          img[b * I:(b + 1) * I])])
        rm = torch.from_numpy(_row_map(T + I, T, B).astype(np.int64)).cuda()
        limit = _limits(T, T + I, geo["text_causal"])
    else:
        B, T, runs = 1, 0, _ti2i_runs(case)
        hidden = torch.cat([(img if is_img else txt)[at:at + n] for n, is_img, at in runs])
        ends, limit = 0, []
        for n, is_img, _ in runs:  # text causal, image runs whole
            r = torch.arange(ends, ends + n, device="cuda") + 1
            ends += n
            limit.append(torch.full_like(r, ends) if is_img else r)
        limit = torch.cat(limit)
        rm = (torch.arange(ends, device="cuda") < ends - runs[-1][0]).long()
    for l in range(case["layers"]):
        hidden = _block64(geo, _weights64(s.dit, geo, seed, l), hidden, mod, rm, cos, sin, limit, B)
    out = _final64(geo, seed, hidden, norm_out, rm)
    return out[-runs[-1][0]:] if kind == "ti2i" else out.view(B, -1, geo["z_dim"])
