"""The work that a user of the library has it do, as measurable cases.

Four kinds of work, each through the public entry points:

  layer  the linears of one decoder layer on a batch of token rows that stay in device memory: the fused
         prep + linear calls of include/eif_hip.h (eif_hip_qlinear_prep, eif_hip_qlinear_prep_glu), one call per
         matrix. Few rows are decoding, many are a prompt. Ternary with group scales (the BitNet layers), ternary with
         one scale a row (TTML and GGUF BitNet files), INT8 (dense row-scaled models).
  int4   the INT4 linears around the vocabulary head: gate|up, down and the tied head.
  model  a whole BitNet model (include/eif_hip_decode.h): reset, prompt, token steps, logits.
  host   the linears of one layer for one token through the drop-in host API, called as the reference's token loop
         calls them (rotate, then one GEMV per matrix, everything in host memory).

Inputs are made from the seed alone. Weights: ternary codes, INT8 and INT4 codes uniform, scales |N(0,1)| times a
constant; activations N(0,1) with 1 % outliers 20 times as large, which is what the absmax quantization meets.
"""
import ctypes as C
import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bitllm.c_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import bitllm_hip as bh  # noqa: E402

_DEV = "cuda:0"
_EPS = 1e-5

# The BitNet-b1.58-2B layer: 20 query and 5 KV heads of 128, g128 scales, g96 in front of the down projection's.
_BITNET_2B = dict(kind="layer", fmt="ternary", dim=2560, q_dim=2560, kv_dim=640, hidden=6912, group=128, group_down=96,
                  wht=128)
# Qwen2.5-0.5B-like INT8 layer: 14 query and 2 KV heads of 64.
_INT8_05B = dict(kind="layer", fmt="int8", dim=896, q_dim=896, kv_dim=128, hidden=4864, group=0, group_down=0, wht=0)
_INT4 = dict(kind="int4", dim=1024, hidden=3584, vocab=151936)
_MODEL = dict(kind="model", layers=30, vocab=128256, context=2048)


def listed():
    return [
        # one decoded token: every launch and every microsecond of a dependent chain counts
        dict(_BITNET_2B, name="bitnet_layer_1", tokens=1),
        # a few users' tokens at once, or drafted tokens being checked
        dict(_BITNET_2B, name="bitnet_layer_24", tokens=24),
        # a prompt
        dict(_BITNET_2B, name="bitnet_layer_512", tokens=512),
        # prompts of several users, or a long document; an odd count
        dict(_BITNET_2B, name="bitnet_layer_3001", tokens=3001),
        # a short prompt on a model with one scale per row and no rotation (TTML and GGUF files)
        dict(_BITNET_2B, name="bitnet_rows_layer_200", tokens=200, group=0, group_down=0, wht=0),
        # a dense INT8 model: one decoded token, and a prompt
        dict(_INT8_05B, name="int8_layer_1", tokens=1),
        dict(_INT8_05B, name="int8_layer_128", tokens=128),
        # an INT4 model's feed-forward and tied vocabulary head: one token, and the last rows of a batch of sequences
        dict(_INT4, name="int4_head_1", tokens=1),
        dict(_INT4, name="int4_head_32", tokens=32),
        # a request to a served model: a prompt of ordinary length, then tokens one by one
        dict(_MODEL, name="model_generate", prompt=511, steps=64),
        # a long prompt of which only the next token is wanted
        dict(_MODEL, name="model_prompt", prompt=1900, steps=1),
        # the drop-in library under the reference's own token loop
        dict(kind="host", name="host_layer", dim=2560, q_dim=2560, kv_dim=640, hidden=6912, group=128, group_down=96,
             wht=128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _group(rng, cols):
    """A group size that a matrix of `cols` columns has in earnest: 128 most often, the others that divide it."""
    fits = [g for g in (32, 64, 96, 256) if cols % g == 0] or [32]
    return 128 if cols % 128 == 0 and rng.random() < 0.6 else rng.choice(fits)


def draw(rng: random.Random):
    kind = rng.choice(["bitnet", "bitnet", "bitnet", "rows", "int8", "int8", "int4", "model", "host"])
    if kind in ("bitnet", "rows", "host"):
        heads, kv = rng.randint(6, 32), rng.randint(1, 8)
        dim, hidden = 128 * heads, 128 * rng.randint(12, 72)
        c = dict(kind="host" if kind == "host" else "layer", dim=dim, q_dim=dim, kv_dim=128 * kv, hidden=hidden,
                 group=_group(rng, dim), group_down=_group(rng, hidden), wht=rng.choice([128, 128, 128, 64, 0]))
        if kind == "host":
            return c
        c["fmt"] = "ternary"
        if kind == "rows":
            c.update(group=0, group_down=0, wht=0)
        most = 3001 * _weights(_BITNET_2B) // _weights(c)
        c["tokens"] = _log_int(rng, 1, min(3001, most))
        return c
    if kind == "int8":
        dim = 64 * rng.randint(8, 40)
        return dict(kind="layer", fmt="int8", dim=dim, q_dim=dim, kv_dim=64 * rng.randint(1, 8),
                    hidden=32 * rng.randint(40, 220), group=0, group_down=0, wht=0, tokens=_log_int(rng, 1, 700))
    if kind == "int4":
        return dict(kind="int4", dim=32 * rng.randint(16, 64), hidden=32 * rng.randint(32, 160),
                    vocab=rng.randint(32000, 151936), tokens=_log_int(rng, 1, 48))
    return dict(kind="model", layers=rng.randint(3, 30), vocab=rng.randint(32000, 128256), context=2048,
                prompt=_log_int(rng, 2, 1900), steps=_log_int(rng, 1, 64))


def _weights(c):
    """Weights of one layer (columns times rows over its matrices)."""
    return sum(r * k for r, k in _layer_shapes(c))


def _layer_shapes(c):
    """(rows, cols) of a layer's matrices: q|k|v, o, gate|up, down."""
    return [(c["q_dim"] + 2 * c["kv_dim"], c["dim"]), (c["dim"], c["q_dim"]), (2 * c["hidden"], c["dim"]),
            (c["dim"], c["hidden"])]


# ---- inputs ----

def _gen(seed):
    return torch.Generator(device=_DEV).manual_seed(int(seed) * 7919 + 13)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=_DEV)


def _activations(g, m, k):
    x = _randn(g, m, k)
    return torch.where(torch.rand((m, k), generator=g, device=_DEV) < 0.01, 20.0 * x, x).contiguous()


def _signs(g, n):
    return torch.randint(0, 2, (n,), generator=g, device=_DEV).float() * 2.0 - 1.0


def _norm_weight(g, n):
    return 1.0 + 0.1 * _randn(g, n)


def _codes(g, fmt, rows, cols):
    """Integer weights [rows, cols] as int8."""
    lo, hi = {"ternary": (-1, 2), "int8": (-127, 128), "int4": (-8, 8)}[fmt]
    return torch.randint(lo, hi, (rows, cols), generator=g, device=_DEV, dtype=torch.int8)


def _pack(fmt, w):
    """The reference's storage of integer weights (cols a multiple of 4)."""
    if fmt == "int8":
        return w
    if fmt == "int4":
        u = (w + 8).to(torch.uint8)
        return ((u[:, 0::2] << 4) | u[:, 1::2]).contiguous()
    c = torch.where(w < 0, 2, w).to(torch.uint8)
    return (c[:, 0::4] | (c[:, 1::4] << 2) | (c[:, 2::4] << 4) | (c[:, 3::4] << 6)).contiguous()


def _scales(g, fmt, rows, cols, group):
    if group:
        return _randn(g, rows, -(-cols // group)).abs() * 0.02 + 0.001
    return _randn(g, rows).abs() * 0.01 + 0.001


def _matrix(g, fmt, rows, cols, group):
    return _codes(g, fmt, rows, cols), _scales(g, fmt, rows, cols, group)


def _layer_inputs(c, seed):
    """The tensors of a layer case: its matrices in order, the token rows, norm weights and rotation signs."""
    g = _gen(seed)
    groups = [c["group"]] * 3 + [c["group_down"]]
    d = {"w": [_matrix(g, c["fmt"], r, k, grp) for (r, k), grp in zip(_layer_shapes(c), groups)], "groups": groups}
    m = c["tokens"]
    d["x"], d["attn"] = _activations(g, m, c["dim"]), _activations(g, m, c["q_dim"])
    # ternary layers form the down projection's input from gate|up; the others are given it
    d["h"] = _activations(g, m, c["hidden"]) if c["fmt"] != "ternary" else None
    d["nw"] = [_norm_weight(g, k) for _, k in _layer_shapes(c)]
    d["signs"] = [_signs(g, k) if c["wht"] else None for _, k in _layer_shapes(c)]
    return d


def _int4_shapes(c):
    return [(2 * c["hidden"], c["dim"]), (c["dim"], c["hidden"]), (c["vocab"], c["dim"])]


def _int4_inputs(c, seed):
    g = _gen(seed)
    d = {"w": [_matrix(g, "int4", r, k, 0) for r, k in _int4_shapes(c)]}
    d["x"] = [_activations(g, c["tokens"], k) for _, k in _int4_shapes(c)]
    d["nw"] = [_norm_weight(g, k) for _, k in _int4_shapes(c)]
    return d


def _model_config(c):
    return dict(dim=2560, hidden=6912, n_layers=c["layers"], n_heads=20, n_kv_heads=5, head_dim=128, vocab=c["vocab"],
                seq_len=c["context"], rope_theta=500000.0, rms_eps=1e-5, sub_eps=1e-5, wht_dim=128, wht_q=128,
                wht_hidden=128, wht_norm_dim=bh.wht_norm(128), wht_norm_q=bh.wht_norm(128),
                wht_norm_hidden=bh.wht_norm(128), g_q=128, g_o=128, g_13=128, g_2=96)


_MODEL_PARTS = ("q", "k", "v", "o", "1", "3", "2")


def _model_shape(part, cfg):
    qd, kvd = cfg["n_heads"] * cfg["head_dim"], cfg["n_kv_heads"] * cfg["head_dim"]
    d, h = cfg["dim"], cfg["hidden"]
    return {"q": (qd, d, cfg["g_q"]), "k": (kvd, d, cfg["g_q"]), "v": (kvd, d, cfg["g_q"]), "o": (d, qd, cfg["g_o"]),
            "1": (h, d, cfg["g_13"]), "3": (h, d, cfg["g_13"]), "2": (d, h, cfg["g_2"])}[part]


def _model_globals(g, cfg):
    d, v = cfg["dim"], cfg["vocab"]
    return {"emb": _codes(g, "int8", v, d), "emb_scale": _randn(g, v).abs() * 0.01 + 0.01,
            "wcls": _codes(g, "int8", v, d), "wcls_scale": _randn(g, v).abs() * 0.01 + 0.002,
            "rms_final": _norm_weight(g, d), "signs_dim": _signs(g, d), "signs_q": _signs(g, cfg["n_heads"] * 128),
            "signs_hidden": _signs(g, cfg["hidden"])}


def _model_layer(seed, layer, cfg):
    g = _gen(seed * 64 + layer + 1)
    w = {p: _matrix(g, "ternary", *_model_shape(p, cfg)) for p in _MODEL_PARTS}
    for p in ("o", "2"):   # what a layer adds to the residual stream starts at 1 / sqrt(2 layers), as trained models do
        w[p] = (w[p][0], w[p][1] / math.sqrt(2.0 * cfg["n_layers"]))
    for name, n in (("rms_att", cfg["dim"]), ("rms_ffn", cfg["dim"]), ("rms_sub_att", cfg["n_heads"] * 128),
                    ("rms_sub_ffn", cfg["hidden"])):
        w[name] = _norm_weight(g, n)
    return w


def _model_ids(c, seed):
    # every token of the prompt and of the steps is given, so that a run's results do not hang on a near tie of two
    # logits of a random model
    return np.random.default_rng(seed).integers(0, c["vocab"], c["prompt"] + c["steps"]).astype(np.int32)


def _host_inputs(c, seed):
    g = _gen(seed)
    rows = {"q": c["q_dim"], "k": c["kv_dim"], "v": c["kv_dim"], "o": c["dim"], "1": c["hidden"], "3": c["hidden"],
            "2": c["dim"]}
    cols = {"o": c["q_dim"], "2": c["hidden"]}
    w = {}
    for p in _MODEL_PARTS:
        k = cols.get(p, c["dim"])
        grp = c["group_down"] if p == "2" else c["group"]
        w[p] = (*_matrix(g, "ternary", rows[p], k, grp), grp)
    ins = [(p, _activations(g, 1, k)[0], _signs(g, k) if c["wht"] else None)
           for p, k in (("qkv", c["dim"]), ("o", c["q_dim"]), ("13", c["dim"]), ("2", c["hidden"]))]
    return w, ins


# ---- what a program has in hand, and one pass ----

class _Linears:
    """Resident weights, rows and output buffers of a list of linear calls, as a program keeps them."""

    def __init__(self):
        self.keep, self.calls, self.out = [], [], []

    def add(self, weight, spec, y, glu=False):
        self.keep += [weight, spec, y]
        self.calls.append((weight.h, spec, C.c_void_p(y.data_ptr()), y.stride(0), y.shape[0], glu))
        self.out.append(y)

    def run(self):
        lib, st = bh.load(), torch.cuda.current_stream().cuda_stream
        for h, spec, y, ldy, m, glu in self.calls:
            rc = lib.eif_hip_qlinear_prep_glu(h, spec, y, ldy, m, st) if glu else \
                lib.eif_hip_qlinear_prep(h, spec, None, y, ldy, m, st)
            if rc:
                bh.check(rc, "linear")
        return self.out


_FMT = {"ternary": bh.W_TERNARY, "int8": bh.W_INT8, "int4": bh.W_INT4}


def _resident(fmt, w, group):
    return bh.QWeight(_FMT[fmt], w[0].shape[0], w[0].shape[1], group, _pack(fmt, w[0]), w[1], on_device=True)


def _empty(m, n):
    return torch.empty((m, n), device=_DEV)


def _prepare_layer(c, seed):
    d, s, m = _layer_inputs(c, seed), _Linears(), c["tokens"]
    w = [_resident(c["fmt"], x, grp) for x, grp in zip(d["w"], d["groups"])]
    norm = bh.wht_norm(c["wht"]) if c["wht"] else 1.0

    def spec(i, x, pre, x2=None):
        s.keep += [x, x2, d["nw"][i], d["signs"][i]]
        return bh.prep_spec(x, pre, x2, d["nw"][i], _EPS, d["signs"][i], c["wht"], norm)

    ternary = c["fmt"] == "ternary"
    s.add(w[0], spec(0, d["x"], bh.PRE_RMS), _empty(m, w[0].rows))
    s.add(w[1], spec(1, d["attn"], bh.PRE_RMS if ternary else bh.PRE_NONE), _empty(m, c["dim"]))
    # up to 8 rows of a g128 layer the decoder's gated call writes SiLU(gate) * up; else gate and up, the SwiGLU in front
    # of the down projection
    glu = _gated(c)
    gu = _empty(m, c["hidden"] * (1 if glu else 2))
    s.add(w[2], spec(2, d["x"], bh.PRE_RMS), gu, glu)
    if not ternary:
        last = spec(3, d["h"], bh.PRE_NONE)
    elif glu:
        last = spec(3, gu, bh.PRE_RMS)
    else:
        last = spec(3, gu[:, :c["hidden"]], bh.PRE_SWIGLU_RMS, gu[:, c["hidden"]:])
    s.add(w[3], last, _empty(m, c["dim"]))
    torch.cuda.synchronize()
    return s


def _gated(c):
    return c["fmt"] == "ternary" and c["tokens"] <= 8 and c["group"] == 128 and c["wht"] in (0, 128)


def _prepare_int4(c, seed):
    d, s = _int4_inputs(c, seed), _Linears()
    for w, x, nw in zip(d["w"], d["x"], d["nw"]):
        s.keep += [x, nw]
        s.add(_resident("int4", w, 0), bh.prep_spec(x, bh.PRE_RMS, None, nw, _EPS), _empty(c["tokens"], w[0].shape[0]))
    torch.cuda.synchronize()
    return s


class _Model:
    def __init__(self, c, seed):
        cfg = _model_config(c)
        w = {k: v.cpu().numpy() for k, v in _model_globals(_gen(seed), cfg).items()}
        layers = []
        for i in range(c["layers"]):
            lw = _model_layer(seed, i, cfg)
            layers.append({("w" + p): _pack("ternary", lw[p][0]).cpu().numpy() for p in _MODEL_PARTS} |
                          {("g" + p): lw[p][1].cpu().numpy() for p in _MODEL_PARTS} |
                          {k: v.cpu().numpy() for k, v in lw.items() if k.startswith("rms")})
        for k in layers[0]:
            w[k] = np.concatenate([x[k] for x in layers])
        self.model = bh.BitnetModel(cfg, w)
        self.ids, self.prompt, self.steps = _model_ids(c, seed), c["prompt"], c["steps"]

    def run(self):
        m = self.model
        m.reset(self.ids)
        m.prefill(self.prompt)
        m.steps(self.steps, graph=True)
        return m.logits()


class _Host:
    def __init__(self, c, seed):
        w, ins = _host_inputs(c, seed)
        self.wht = c["wht"]
        self.w = {p: (_pack("ternary", a).cpu().numpy(), s.cpu().numpy(), grp) for p, (a, s, grp) in w.items()}
        self.ins = [(p, x.cpu().numpy(), None if s is None else s.cpu().numpy()) for p, x, s in ins]
        self.rot = [np.empty_like(x) for _, x, _ in self.ins]
        self.out = {p: np.empty(a.shape[0], np.float32) for p, (a, _, _) in self.w.items()}

    def run(self):
        lib = bh.load()
        for (parts, x, signs), r in zip(self.ins, self.rot):
            np.copyto(r, x)
            if self.wht:
                lib.eif_hadamard_rotate_f32(bh.ptr(r), bh.ptr(signs), r.size, self.wht)
            for p in parts:
                a, s, grp = self.w[p]
                lib.eif_matmul_bitnet_block_f32(bh.ptr(a), bh.ptr(s), grp, bh.ptr(r), None, bh.ptr(self.out[p]),
                                                a.shape[0], r.size)
        return self.out

    def __del__(self):
        # the library keeps device copies by host address: a program drops them before it frees the memory
        try:
            for a, s, _ in self.w.values():
                bh.load().eif_hip_forget_host_weights(bh.ptr(a))
                bh.load().eif_hip_forget_host_weights(bh.ptr(s))
        except Exception:
            pass


def prepare(case, seed):
    bh.check(bh.load().eif_hip_init(0), "eif_hip_init")
    return {"layer": _prepare_layer, "int4": _prepare_int4, "model": _Model, "host": _Host}[case["kind"]](case, seed)


def run(state):
    return state.run()


# ---- work ----

def _code_bytes(fmt, rows, cols):
    return rows * -(-cols * {"ternary": 2, "int4": 4, "int8": 8}[fmt] // 8)


def _scale_bytes(rows, cols, group):
    return 4 * rows * (-(-cols // group) if group else 1)


def work(case):
    c = case
    if c["kind"] == "layer":
        m, shapes = c["tokens"], _layer_shapes(c)
        groups = [c["group"]] * 3 + [c["group_down"]]
        b = sum(_code_bytes(c["fmt"], r, k) + _scale_bytes(r, k, g) for (r, k), g in zip(shapes, groups))
        out = [r for r, _ in shapes]
        if _gated(c):
            out[2] //= 2
        ins = c["dim"] + c["q_dim"] + (0 if c["fmt"] == "ternary" else c["hidden"])
        return {"bytes": b + 4 * m * (ins + sum(out)), "flops": 2 * m * _weights(c)}
    if c["kind"] == "int4":
        m, shapes = c["tokens"], _int4_shapes(c)
        return {"bytes": sum(_code_bytes("int4", r, k) + 4 * r + 4 * m * (r + k) for r, k in shapes),
                "flops": 2 * m * sum(r * k for r, k in shapes)}
    if c["kind"] == "host":
        shapes = {p: (a, b, c["group_down"] if p == "2" else c["group"]) for p, a, b in
                  (("q", c["q_dim"], c["dim"]), ("k", c["kv_dim"], c["dim"]), ("v", c["kv_dim"], c["dim"]),
                   ("o", c["dim"], c["q_dim"]), ("1", c["hidden"], c["dim"]), ("3", c["hidden"], c["dim"]),
                   ("2", c["dim"], c["hidden"]))}
        b = sum(_code_bytes("ternary", r, k) + _scale_bytes(r, k, g) + 4 * r for r, k, g in shapes.values())
        return {"bytes": b + 4 * (2 * c["dim"] + c["q_dim"] + c["hidden"]),
                "flops": 2 * sum(r * k for r, k, _ in shapes.values())}
    cfg = dict(dim=2560, hidden=6912, n_heads=20, n_kv_heads=5, head_dim=128, g_q=128, g_o=128, g_13=128, g_2=96)
    shapes = [_model_shape(p, cfg) for p in _MODEL_PARTS]
    layers = c["layers"] * sum(_code_bytes("ternary", r, k) + _scale_bytes(r, k, g) for r, k, g in shapes)
    head = c["vocab"] * (cfg["dim"] + 4)
    kv = c["layers"] * 2 * 2 * 5 * 128   # bytes of one position's keys and values
    p, t = c["prompt"], c["steps"]
    mean = p + (t + 1) / 2
    params = c["layers"] * sum(r * k for r, k, _ in shapes)
    attn = c["layers"] * 4 * 2560 * (p * (p + 1) / 2 + t * mean)
    return {"bytes": int((1 + t) * (layers + head) + kv * (p + t * mean)),
            "flops": int(2 * params * (p + t) + 2 * (1 + t) * c["vocab"] * cfg["dim"] + attn)}


# ---- tolerances ----

def tolerance(case):
    """Measured against `exact`, about four times what was seen. The linears are exact integer sums with FP32 scales
    (3e-7), but an activation on a rounding boundary of its INT8 code may take the neighbouring code: in a batch of many
    rows a few do (4.4e-4 in the down projection, whose input is itself computed). In a model such a code travels
    through every later layer (2.3e-2 in the logits of 30 layers). The host calls take FP32 activations (2.7e-7)."""
    return {"rel": {"host": 1.2e-6, "model": 0.09}.get(case["kind"], 2e-3)}


# ---- the same results in 64 bits ----

def _rotate(v, block, norm):
    """Blockwise Walsh-Hadamard transform of the last axis."""
    if not block:
        return v
    h = torch.ones((1, 1), dtype=torch.float64, device=v.device)
    while h.shape[0] < block:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return ((v.reshape(-1, block) @ h) * norm).reshape(v.shape)


def _rms(v, eps, w):
    return v / torch.sqrt((v * v).mean(-1, keepdim=True) + eps) * w.double()


def _quant_rows(v):
    """Absmax INT8 codes and scales of every row, round half away from zero."""
    a = v.abs().amax(-1, keepdim=True)
    t = v * (127.0 / a)
    return torch.trunc(t + torch.copysign(torch.full_like(t, 0.5), t)).clamp(-128, 127), a / 127.0


def _dense(w, scales, group):
    """Integer weights times their scales in float64."""
    w = w.double()
    if not group:
        return w * scales.double()[:, None]
    return w * scales.double().repeat_interleave(group, 1)[:, :w.shape[1]]


def _linear(v, w, scales, group, signs=None, wht=0, norm=1.0):
    """The quantized linear on float64 rows v (already through the pre-op)."""
    if wht and signs is not None:
        v = v * signs.double()
    q, s = _quant_rows(_rotate(v, wht, norm))
    return (q * s) @ _dense(w, scales, group).t()


def _silu(g):
    return g / (1.0 + torch.exp(-g))


def _exact_layer(c, seed):
    d = _layer_inputs(c, seed)
    norm = bh.wht_norm(c["wht"]) if c["wht"] else 1.0
    ternary = c["fmt"] == "ternary"

    def lin(i, v):
        return _linear(v, *d["w"][i], d["groups"][i], d["signs"][i], c["wht"], norm)

    def normed(i, v):
        return _rms(v, _EPS, d["nw"][i])

    x, a = d["x"].double(), d["attn"].double()
    gu = lin(2, normed(2, x))
    h = _silu(gu[:, :c["hidden"]]) * gu[:, c["hidden"]:]
    down = lin(3, normed(3, h)) if ternary else lin(3, d["h"].double())
    return [lin(0, normed(0, x)), lin(1, normed(1, a) if ternary else a), h if _gated(c) else gu, down]


def _exact_int4(c, seed):
    d = _int4_inputs(c, seed)
    out = []
    for (w, s), x, nw in zip(d["w"], d["x"], d["nw"]):
        q, xs = _quant_rows(_rms(x.double(), _EPS, nw))
        step = 16384   # rows at a time: the head in float64 is large
        out.append(torch.cat([(q * xs) @ _dense(w[i:i + step], s[i:i + step], 0).t() for i in range(0, w.shape[0], step)], 1))
    return out


def _exact_host(c, seed):
    w, ins = _host_inputs(c, seed)
    norm = bh.wht_norm(c["wht"]) if c["wht"] else 1.0
    out = {}
    for parts, x, signs in ins:
        v = x.double()
        if c["wht"]:
            v = _rotate(v * signs.double(), c["wht"], norm)
        for p in parts:
            a, s, grp = w[p]
            out[p] = (_dense(a, s, grp) @ v).cpu().numpy()
    return {p: out[p] for p in _MODEL_PARTS}


def _exact_model(c, seed):
    cfg = _model_config(c)
    gl = _model_globals(_gen(seed), cfg)
    ids = torch.from_numpy(_model_ids(c, seed)).long().to(_DEV)
    n, hd, nh, nkv = len(ids), 128, cfg["n_heads"], cfg["n_kv_heads"]
    norm = cfg["wht_norm_dim"]
    x = gl["emb"][ids].double() * gl["emb_scale"][ids].double()[:, None]
    ang = torch.arange(n, device=_DEV).double()[:, None] / \
        cfg["rope_theta"] ** (torch.arange(hd // 2, device=_DEV).double() * 2 / hd)
    cos, sin = torch.cos(ang)[:, None], torch.sin(ang)[:, None]

    def rope(v):
        a, b = v[..., :hd // 2], v[..., hd // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    mask = torch.ones((n, n), dtype=torch.bool, device=_DEV).triu(1)
    for i in range(c["layers"]):
        w = _model_layer(seed, i, cfg)

        def lin(p, v, signs):
            return _linear(v, *w[p], _model_shape(p, cfg)[2], gl[signs], 128, norm)

        v = _rms(x, cfg["rms_eps"], w["rms_att"])
        q = rope(lin("q", v, "signs_dim").reshape(n, nh, hd))
        k = rope(lin("k", v, "signs_dim").reshape(n, nkv, hd)).half().double()   # the cache holds fp16
        val = lin("v", v, "signs_dim").reshape(n, nkv, hd).half().double()
        att = torch.empty((n, nh, hd), dtype=torch.float64, device=_DEV)
        for h in range(nh):
            g = h // (nh // nkv)
            s = (q[:, h] @ k[:, g].t().contiguous()) / math.sqrt(hd)
            att[:, h] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ val[:, g]
        x = x + lin("o", _rms(att.reshape(n, nh * hd), cfg["sub_eps"], w["rms_sub_att"]), "signs_q")
        v = _rms(x, cfg["rms_eps"], w["rms_ffn"])
        h = _silu(lin("1", v, "signs_dim")) * lin("3", v, "signs_dim")
        x = x + lin("2", _rms(h, cfg["sub_eps"], w["rms_sub_ffn"]), "signs_hidden")
    q, s = _quant_rows(_rms(x[-1:], cfg["rms_eps"], gl["rms_final"]))
    step = 16384
    out = [(q * s) @ _dense(gl["wcls"][i:i + step], gl["wcls_scale"][i:i + step], 0).t() for i in range(0, cfg["vocab"], step)]
    return torch.cat(out, 1)[0].cpu().numpy()


def exact(case, seed):
    f = {"layer": _exact_layer, "int4": _exact_int4, "model": _exact_model, "host": _exact_host}[case["kind"]]
    return f(case, seed)
