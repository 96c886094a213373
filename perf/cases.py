"""Performance cases of this framework: what a program that generates audio with
it has the GPU do, from single graph nodes to whole model calls.

A 9 s clip is 194 latent, 77 text, 72 clip and 216 sync frames, a 30 s one 646,
77, 240 and 720; classifier-free guidance makes every step a batch of 2. The
nodes go through the C entry points of libtsk.so with descriptors that are
built once (as a ggml backend holds them), the models through the front end's
device entry points. Device memory is torch's; both use the null stream.
"""
import ctypes
import math

import numpy as np
import torch

from __graft_entry__ import load_tsk

DEV = "cuda"
# (inputs, outputs) of the models' linear layers: latent / sync / clip input,
# attention and MLP projections, adaLN, SwiGLU halves, T5
LINEAR = [(64, 1024), (768, 1024), (1024, 1024), (1024, 2816), (1024, 3072), (1024, 4096), (1024, 6144), (2048, 1024),
          (2048, 2048), (2816, 1024), (4096, 1024)]


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # QK-RMSNorm + RoPE of one layer's queries at 9 s: a few microseconds of work
        {"name": "qk_norm_rope_9s", "kind": "qk_norm_rope", "batch": 2, "seq": 194},
        # the adaLN modulation of one block: two conditioning rows against 12 MB of weights
        {"name": "linear_bf16_adaln", "kind": "linear", "type": "bf16", "act": "f32", "rows": 2, "k": 1024, "m": 6144},
        # the QKV projection of a fused block at 9 s
        {"name": "linear_bf16_9s", "kind": "linear", "type": "bf16", "act": "f32", "rows": 388, "k": 1024, "m": 3072},
        # the QKV projection of a joint block at 30 s with a quantized file's weights
        {"name": "linear_q8_0_30s", "kind": "linear", "type": "q8_0", "act": "f32", "rows": 1446, "k": 1024, "m": 3072},
        # the k3 output projection of a quantized file, whose convolution kernels stay F32
        {"name": "conv_f32_30s", "kind": "conv", "type": "f32", "batch": 2, "seq": 646, "ic": 1024, "oc": 1024, "kw": 3},
        # the SwiGLU convolution MLP of a latent block at 30 s
        {"name": "conv_mlp_bf16_30s", "kind": "conv_mlp", "type": "bf16", "batch": 2, "seq": 646},
        # joint attention over latent and text tokens at 9 s
        {"name": "attention_9s", "kind": "attention", "type": "f16", "batch": 2, "n": 271},
        # joint attention over latent, clip and text tokens at 30 s
        {"name": "attention_30s", "kind": "attention", "type": "f16", "batch": 2, "n": 1040},
        # text encoding of a full 512-token prompt, two of the encoder's layers
        {"name": "t5_512", "kind": "t5", "tokens": 512, "padded": 64},
        # decoding a 30 s latent to stereo audio
        {"name": "vae_30s", "kind": "vae", "frames": 646},
        # one whole flow step of the 21-block transformer at 9 s
        {"name": "dit_step_9s", "kind": "dit", "batch": 2, "frames": 194},
        # one flow step of the three-stream graph at 9 s, quantized file's types (2 joint + 1 fused block)
        {"name": "graph_q8_0_9s", "kind": "graph", "type": "q8_0", "batch": 2, "seconds": 9},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["qk_norm_rope", "linear", "linear", "conv", "conv_mlp", "attention", "t5", "vae", "dit", "graph"])
    b = rng.choice([1, 2])
    if kind == "qk_norm_rope":
        return {"kind": kind, "batch": b, "seq": _log(rng, 16, 646)}
    if kind == "linear":
        k, m = rng.choice(LINEAR)
        return {"kind": kind, "type": rng.choice(["bf16", "q8_0", "f32"]), "act": rng.choice(["f32", "f32", "bf16"]),
                "rows": _log(rng, 1, 2080), "k": k, "m": m}
    if kind == "conv":
        ic, oc, kw = rng.choice([(1024, 1024, 3), (768, 1024, 7), (1024, 64, 7), (64, 1024, 3)])
        return {"kind": kind, "type": rng.choice(["bf16", "f32"]), "batch": b, "seq": _log(rng, 16, 720), "ic": ic,
                "oc": oc, "kw": kw}
    if kind == "conv_mlp":
        return {"kind": kind, "type": rng.choice(["bf16", "f32"]), "batch": b, "seq": _log(rng, 16, 646)}
    if kind == "attention":
        return {"kind": kind, "type": rng.choice(["f16", "bf16"]), "batch": b, "n": _log(rng, 16, 1040)}
    if kind == "t5":
        n = _log(rng, 8, 512)
        return {"kind": kind, "tokens": n, "padded": rng.randrange(n // 2 + 1)}
    if kind == "vae":
        return {"kind": kind, "frames": _log(rng, 4, 640)}
    if kind == "dit":
        return {"kind": kind, "batch": b, "frames": _log(rng, 16, 646)}
    return {"kind": kind, "type": rng.choice(["q8_0", "bf16"]), "batch": b, "seconds": rng.randint(2, 30)}


# ---------------------------------------------------------------- inputs
class _Rand:
    """seeded inputs, made on the GPU"""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(1 + int(seed))

    def __call__(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device=DEV, dtype=torch.float32) * std


def _tsk():
    t = load_tsk()
    t.init(0)
    return t


def _q8_blocks(w):
    """f32 rows as ggml Q8_0 blocks (M, K / 32, 34) and the values they hold (f64)"""
    m, k = w.shape
    b = w.reshape(m, k // 32, 32)
    d = (b.abs().amax(-1, keepdim=True) / 127.0).half()
    q = torch.where(d > 0, torch.round(b / d.float()), torch.zeros_like(b)).clamp(-127, 127).to(torch.int8)
    blocks = torch.cat([d.view(torch.uint8), q.view(torch.uint8)], dim=-1).contiguous()
    return blocks, (q.double() * d.double()).reshape(m, k)


def _weight(r, typ, *shape, std):
    w = r(*shape, std=std)
    return w.bfloat16() if typ == "bf16" else w


def _kernel(r, typ, oc, ic, kw):
    """a convolution kernel laid out kw-major once (tsk_conv1d_pack_weight's layout), seen as (OC, IC, KW)"""
    return _weight(r, typ, oc, kw, ic, std=(ic * kw) ** -0.5).permute(0, 2, 1)


def _type(t, x):
    return {torch.float32: t.F32, torch.float16: t.F16, torch.bfloat16: t.BF16, torch.int32: t.I32}[x.dtype]


def _descs(t, *xs):
    return [None if x is None else t.desc(x, _type(t, x)) for x in xs]


def _op(t, name, *args):
    """a prepared call of a C entry point on the null stream"""
    fn, keep = getattr(t.load(), name), args
    refs = tuple(ctypes.byref(a) if isinstance(a, t.TskTensor) else a for a in keep)

    def call():
        rc = fn(*refs, None)
        if rc:
            t.check(rc)
    return call


def _tensors(case, seed):
    """a node's operands"""
    r, kind = _Rand(seed), case["kind"]
    if kind == "qk_norm_rope":
        return {"x": r(case["batch"], case["seq"], 16, 64), "w": 1 + r(64, std=0.1),
                "pos": torch.arange(case["seq"], device=DEV, dtype=torch.int32)}
    if kind == "linear":
        x = r(case["rows"], case["k"])
        s = {"x": x.bfloat16() if case["act"] == "bf16" and case["type"] == "bf16" else x, "bias": r(case["m"], std=0.02)}
        if case["type"] == "q8_0":
            s["blocks"], s["values"] = _q8_blocks(r(case["m"], case["k"], std=case["k"] ** -0.5))
        else:
            s["w"] = _weight(r, case["type"], case["m"], case["k"], std=case["k"] ** -0.5)
        return s
    if kind == "conv":
        return {"x": r(case["batch"], case["seq"], case["ic"]), "w": _kernel(r, case["type"], case["oc"], case["ic"], case["kw"]),
                "bias": r(case["oc"], std=0.02)}
    if kind == "conv_mlp":
        return {"x": r(case["batch"], case["seq"], 1024), "w1": _kernel(r, case["type"], 2816, 1024, 3),
                "w3": _kernel(r, case["type"], 2816, 1024, 3), "w2": _kernel(r, case["type"], 1024, 2816, 3)}
    b, n, f = case["batch"], case["n"], torch.float16 if case["type"] == "f16" else torch.bfloat16
    q = r(b, 16, n, 64)
    return {"q": q if case["type"] == "f16" else q.to(f), "k": r(b, 16, n, 64).to(f), "v": r(b, 16, n, 64).to(f)}


# models: the weights are part of the program, the same for every input
_models = {}


def _model_weights(tensors, seed=1234, std=0.02):
    """{name: f32 tensor on the GPU}: matrices N(0, std), rounded to bf16 where they are stored so, norm weights about 1"""
    t, r, out = _tsk(), _Rand(seed), {}
    for name, ne, *typ in tensors:
        shape = [int(x) for x in reversed(ne)]
        while len(shape) > 1 and shape[0] == 1:
            shape = shape[1:]
        w = r(*shape, std=1.0 if name.startswith("empty_") else std)
        if name.endswith("norm.weight"):
            w = 1 + w
        out[name] = w.bfloat16().float() if len(shape) > 1 and typ in ([], [t.BF16]) else w
    return out


def _make_dit(t):
    m = t.Dit(t.dit_config(max_latent=646))
    ws = _model_weights(m.tensors())
    for k, w in ws.items():
        m.set_tensor(k, w.cpu().numpy())
    return m, {k: w.bfloat16() if w.dim() > 1 else w for k, w in ws.items()}


def _make_graph(t, typ):
    m = t.MMDit(t.mmdit_config(depth=3, fused_depth=1, weight_type=t.Q8_0 if typ == "q8_0" else t.BF16))
    ws = _model_weights(m.tensors())
    for name, _, ty in m.tensors():
        if ty == t.Q8_0:
            blocks, values = _q8_blocks(ws[name])
            m.set_tensor_q8_0(name, blocks.cpu().numpy())
            ws[name] = values.float()                      # 8-bit times 11-bit: exact in f32
        else:
            m.set_tensor(name, ws[name].cpu().numpy())
    return m, ws


def _make_vae(t):
    v = t.Vae(t.vae_config(max_latent=646))
    ws = t.vae_synthetic_weights(v.tensors(), seed=77, snake_std=0.1)
    for k, w in ws.items():
        v.set_tensor(k, w)
    return v, {k: torch.from_numpy(np.ascontiguousarray(w)).to(DEV) for k, w in ws.items()}


def _make_t5(t):
    m, r, ws = t.T5(t.t5_config(n_layers=2)), _Rand(44), {}
    for name, ne, ty in m.tensors():
        if ty == t.Q8_0:
            # trained T5 keeps q.k small (it has no softmax scale): q and k at 8^-1/2 of unit variance
            std = ne[0] ** -0.5 * (8 ** -0.5 if name.endswith((".q", ".k")) else 1.0)
            blocks, ws[name] = _q8_blocks(r(int(ne[1]), int(ne[0]), std=std))
            m.set_tensor(name, blocks.cpu().numpy())
        else:
            w = r(int(ne[1]), int(ne[0])) if name == "rel_bias" else 1 + r(int(ne[0]), std=0.1)
            m.set_tensor(name, w.cpu().numpy())
            ws[name] = w
    return m, ws


def _model(kind, typ=None):
    if (kind, typ) not in _models:
        t = _tsk()
        _models[kind, typ] = {"dit": _make_dit, "vae": _make_vae, "t5": _make_t5}[kind](t) if typ is None else _make_graph(t, typ)
    return _models[kind, typ]


def _model_inputs(case, seed):
    r, kind = _Rand(seed), case["kind"]
    if kind == "t5":
        ids = np.arange(1, case["tokens"] + 1, dtype=np.int32)
        if case["padded"]:
            ids[-case["padded"]:] = 0
        return {"x": r(case["tokens"], 2048), "ids": ids}
    if kind == "vae":
        return {"latent": r(64, case["frames"])}
    b = case["batch"]
    t = np.random.default_rng(int(seed)).uniform(0.05, 1.0, 1).astype(np.float32).repeat(b)
    if kind == "dit":
        return {"latent": r(b, 64, case["frames"]), "t": t, "text": r(b, 77, 1024)}
    s = case["seconds"]
    return {"latent": r(b, 64, round(21.533 * s)), "t": t, "clip": r(b, 8 * s, 1024), "sync": r(b, 24 * s, 768),
            "text": r(b, 77, 1024), "t5": r(b, 77, 2048), "g": r(b, 1024)}


def prepare(case, seed):
    t, kind = _tsk(), case["kind"]
    if kind in ("t5", "vae", "dit", "graph"):
        m = _model(kind, case.get("type"))[0]
        s = _model_inputs(case, seed)
        if kind == "t5":
            s["out"] = torch.empty_like(s["x"])
            s["call"] = lambda: m.encode_device(s["x"], s["ids"], s["out"])
        elif kind == "vae":
            s["out"] = torch.empty(2, case["frames"] * m.hop, device=DEV)
            s["call"] = lambda: m.decode_device(s["latent"], s["out"])
        else:
            s["out"] = torch.empty(case["batch"], s["latent"].shape[2], 64, device=DEV)
            rest = (s["text"],) if kind == "dit" else (s["clip"], s["sync"], s["text"], s["t5"], s["g"])
            s["call"] = lambda: m.forward_device(s["latent"], s["t"], *rest, s["out"])
        return s
    s = _tensors(case, seed)
    if kind == "qk_norm_rope":
        s["out"] = torch.empty_like(s["x"])
        x, w, pos, y = _descs(t, s["x"], s["w"], s["pos"], s["out"])
        s["call"] = _op(t, "tsk_qk_norm_rope", x, w, pos, 1e-6, 64, 10000.0, 1.0, y)
    elif kind == "linear":
        s["out"] = torch.empty(case["rows"], case["m"], device=DEV)
        x, bias, y = _descs(t, s["x"], s["bias"], s["out"])
        if case["type"] == "q8_0":                          # repacked once, as a loaded file's weights are
            del s["values"]
            buf = torch.empty(t.load().tsk_q8_0_split_nbytes(case["k"], case["m"]), dtype=torch.uint8, device=DEV)
            s["w"] = t.SplitQ8(buf, case["k"], case["m"])
            w = t.desc(s["w"], t.Q8_0_SPLIT)
            _op(t, "tsk_q8_0_repack", t.desc(s.pop("blocks"), t.Q8_0), w)()
            torch.cuda.synchronize()
        else:
            w, = _descs(t, s["w"])
        s["call"] = _op(t, "tsk_mul_mat", w, x, bias, y)
    elif kind == "conv":
        s["out"] = torch.empty(case["batch"], case["seq"], case["oc"], device=DEV)
        w, bias, x, y = _descs(t, s["w"], s["bias"], s["x"], s["out"])
        s["call"] = _op(t, "tsk_conv1d", w, bias, x, 1, case["kw"] // 2, 1, y)
    elif kind == "conv_mlp":
        s["out"] = torch.empty(case["batch"], case["seq"], 1024, device=DEV)
        s["call"] = _op(t, "tsk_conv_mlp_swiglu", *_descs(t, s["w1"], s["w3"], s["w2"], s["x"], s["out"]))
    else:
        s["out"] = torch.empty(case["batch"], case["n"], 16, 64, device=DEV)
        q, k, v, y = _descs(t, s["q"], s["k"], s["v"], s["out"])
        s["call"] = _op(t, "tsk_flash_attn_ext", q, k, v, None, 0.125, 0.0, 0.0, t.PREC_F32, y)
    return s


def run(state):
    state["call"]()
    return state["out"]


# ---------------------------------------------------------------- what a pass cannot do without
def _vae_layers(frames):
    """(output positions, products per position, weights) of every convolution of the decoder"""
    rows = [(frames, 7 * 64 * 2048, 7 * 64 * 2048)]
    c = 2048
    for s, o in ((8, 1024), (8, 512), (4, 256), (4, 128), (2, 128)):
        frames *= s
        rows.append((frames, 2 * c * o, 2 * s * c * o))
        rows += [(frames, 8 * o * o, 8 * o * o)] * 3
        c = o
    return rows + [(frames, 7 * 128 * 2, 7 * 128 * 2)]


def _swiglu_conv(rows, ic=1024, hid=2816, oc=1024, kw=3):
    return rows * kw * hid * (2 * ic + oc), kw * hid * (2 * ic + oc)


def _work_graph(case):
    """(products, weights) of the 2 joint + 1 fused graph"""
    b, s, h = case["batch"], case["seconds"], 1024
    T, c, y, x = round(21.533 * s), 8 * s, 24 * s, 154
    p = w = 0
    for rows, per in ((b * T, 3 * 64 * h), (b * c, 1024 * h), (b * y, 7 * 768 * h), (b * x, 2048 * h), (b * T, 7 * h * 64),
                      (b, 7 * h * h), (b * T, 6 * 3 * h * h + 2 * h * h), (b, 16 * h * h)):
        p, w = p + rows * per, w + per
    for rows in (T, c, y):
        q = _swiglu_conv(b * rows)
        p, w = p + q[0], w + q[1]
    for rows, conv in ((T, 3), (T, 3), (T, 3), (c, 3), (x, 1)):   # blocks that run whole
        q = _swiglu_conv(b * rows, kw=conv)
        p, w = p + b * rows * (3 + conv) * h * h + q[0], w + (3 + conv) * h * h + q[1]
    p, w = p + b * (c + x) * 3 * h * h, w + 6 * h * h            # the last joint block's clip and text qkv
    n = T + c + x
    return p + b * h * (2 * 2 * n * n + 2 * T * T), w


def work(case):
    kind = case["kind"]
    if kind == "qk_norm_rope":
        n = case["batch"] * case["seq"] * 1024
        return {"bytes": 8 * n, "flops": 10 * n}
    if kind == "linear":
        n, k, m = case["rows"], case["k"], case["m"]
        per = {"bf16": 2, "q8_0": 34 / 32, "f32": 4}[case["type"]]
        act = 2 if case["act"] == "bf16" and case["type"] == "bf16" else 4
        return {"bytes": per * k * m + act * n * k + 4 * n * m, "flops": 2 * n * k * m}
    per = 2 if case.get("type") == "bf16" else 4
    if kind == "conv":
        n, ic, oc, kw = case["batch"] * case["seq"], case["ic"], case["oc"], case["kw"]
        return {"bytes": per * ic * oc * kw + 4 * n * (ic + oc), "flops": 2 * n * ic * oc * kw}
    if kind == "conv_mlp":
        n = case["batch"] * case["seq"]
        p, w = _swiglu_conv(n)
        return {"bytes": per * w + 8 * n * 1024, "flops": 2 * p}
    if kind == "attention":
        b, n = case["batch"], case["n"]
        return {"bytes": b * 16 * n * 64 * (4 + 2 + 2 + 4 if case["type"] == "f16" else 2 + 2 + 2 + 4), "flops": 4 * b * 16 * n * n * 64}
    if kind == "t5":
        n = case["tokens"]
        w = 4 * 2048 * 2048 + 3 * 2048 * 5120
        return {"bytes": 2 * w * 34 / 32 + 8 * n * 2048, "flops": 2 * (2 * n * w + 4 * n * n * 2048)}
    if kind == "vae":
        rows = _vae_layers(case["frames"])
        return {"bytes": 4 * sum(x[2] for x in rows) + 4 * case["frames"] * (64 + 2 * 2048), "flops": 2 * sum(n * p for n, p, _ in rows)}
    if kind == "dit":
        b, T, h = case["batch"], case["frames"], 1024
        lat, txt, adaln = 21 * 12 * h * h, (7 * 3 + 6 * 9) * h * h, (21 * 6 + 6 * 6 + 2 + 2) * h * h
        p = b * (T * (lat + 2 * 64 * h) + 77 * txt + adaln + 2 * h * h)
        at = b * 2 * h * (7 * (T + 77) ** 2 + 14 * T * T)
        return {"bytes": 2 * (lat + txt + adaln + 2 * h * h) + 4 * b * (2 * T * 64 + 77 * h), "flops": 2 * (p + at)}
    p, w = _work_graph(case)
    s = case["seconds"]
    return {"bytes": (2 if case["type"] == "bf16" else 34 / 32) * w + 4 * case["batch"] * (2 * 64 * 22 * s + 8 * s * 1024 + 24 * s * 768 + 77 * 3072),
            "flops": 2 * p}


def tolerance(case):
    """about four times the error against exact() (1e-6 for 32-bit products, 1.7e-3 where activations are rounded to
    bf16, 5e-3 where they are quantized, 3e-4 for attention, 1.2e-4 through the decoder's 37 convolutions)"""
    kind, typ = case["kind"], case.get("type")
    if kind == "qk_norm_rope":
        return {"rel": 1e-5}
    if kind in ("linear", "conv", "conv_mlp"):
        return {"rel": 1e-5 if typ == "f32" else 1e-2 if typ == "bf16" else 2e-2}
    if kind == "attention":
        return {"rel": 1.5e-3 if typ == "f16" else 5e-3}
    if kind == "vae":
        return {"rel": 5e-4}
    return {"rel": 1e-2 if kind == "dit" else 3e-2}


# ---------------------------------------------------------------- the same in 64 bits
def _angles(n, scale=1.0, dims=64, base=10000.0):
    """ggml's RoPE angles: a running product in 32 bits"""
    step = np.float32(base ** np.float32(-2.0 / dims))
    th, out = np.arange(n, dtype=np.float32), []
    for _ in range(dims // 2):
        out.append((th * np.float32(scale)).astype(np.float64))
        th = th * step
    return torch.from_numpy(np.stack(out, -1)).to(DEV)


def _rope(x, ang):
    """x (..., S, H, 64)"""
    z = torch.view_as_complex(x.reshape(*x.shape[:-1], 32, 2).contiguous()) * torch.polar(torch.ones_like(ang), ang)[:, None, :]
    return torch.view_as_real(z).reshape(x.shape)


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _ln(x):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5)


def _attend(q, k, v, scale, bias=None):
    """(B, H, N, D)"""
    s = torch.matmul(q * scale, k.transpose(-1, -2).contiguous())
    if bias is not None:
        s = s + bias
    return torch.matmul(torch.softmax(s, -1), v)


def _conv(x, w, pad, dil=1):
    """x (..., T, IC), w (OC, IC, KW): a sum of shifted products"""
    kw = w.shape[2]
    t = x.shape[-2] + 2 * pad - dil * (kw - 1)
    x = torch.nn.functional.pad(x, (0, 0, pad, pad))
    y = 0
    for i in range(kw):
        y = y + x[..., i * dil:i * dil + t, :] @ w[:, :, i].double().T.contiguous()
    return y


def _silu(x):
    return x / (1 + torch.exp(-x))


def _swiglu(x, w1, w3, w2):
    f = (lambda a, w: _conv(a, w, 1)) if w1.dim() == 3 else (lambda a, w: a @ w.double().T)
    return f(_silu(f(x, w1)) * f(x, w3), w2)


def _exact_node(case, seed):
    s, kind = _tensors(case, seed), case["kind"]
    d = {k: v.double() for k, v in s.items() if k != "blocks"}
    if kind == "qk_norm_rope":
        return _rope(_rms(d["x"], d["w"], 1e-6), _angles(case["seq"]))
    if kind == "linear":
        return d["x"] @ (d["values"] if case["type"] == "q8_0" else d["w"]).T + d["bias"]
    if kind == "conv":
        return _conv(d["x"], s["w"], case["kw"] // 2) + d["bias"]
    if kind == "conv_mlp":
        return _swiglu(d["x"], s["w1"], s["w3"], s["w2"])
    return _attend(d["q"], d["k"], d["v"], 0.125).permute(0, 2, 1, 3).contiguous()


def _snake(x, w, p):
    return x + torch.sin(x * torch.exp(w[p + ".alpha"].double())) ** 2 * torch.exp(-w[p + ".beta"].double())


def _exact_vae(w, latent):
    def conv(x, p, pad, dil=1):
        y = _conv(x, w[p + ".weight"], pad, dil)
        return y + w[p + ".bias"].double() if p + ".bias" in w else y

    x = conv(latent.double().T.contiguous(), "decoder.layers.0", 3)
    for n, s in enumerate((8, 8, 4, 4, 2)):
        bp = "decoder.layers.%d.layers." % (n + 1)
        x, wt = _snake(x, w, bp + "0"), w[bp + "1.weight"]
        y = torch.zeros(x.shape[0], s, wt.shape[0], dtype=torch.float64, device=DEV)
        xp = torch.nn.functional.pad(x, (0, 0, 2, 2))
        for r in range(s):                                  # zero-stuffed input, flipped kernel, padding K - 1 - s / 2
            for k in range(2 * s):
                at = r + k - (2 * s - 1 - s // 2)
                if at % s == 0:
                    y[:, r] += xp[2 + at // s:2 + at // s + x.shape[0]] @ wt[:, :, k].double().T.contiguous()
        x = y.reshape(-1, wt.shape[0]) + w[bp + "1.bias"].double()
        del y, xp
        for u, dil in enumerate((1, 3, 9)):
            rp = bp + "%d.layers." % (u + 2)
            x = x + conv(_snake(conv(_snake(x, w, rp + "0"), rp + "1", 3 * dil, dil), w, rp + "2"), rp + "3", 0)
    return conv(_snake(x, w, "decoder.layers.6"), "decoder.layers.7", 3).T.contiguous()


def _bucket(rel):
    """T5's relative-position bucket: 16 to each side, exact below 8, logarithmic up to 128"""
    a = rel.abs()
    far = (8 + torch.floor(torch.log(a.clamp(min=8).double() / 8) / math.log(16) * 8 + 1e-9).long()).clamp(max=15)
    return torch.where(rel > 0, 16, 0) + torch.where(a < 8, a, far)


def _exact_t5(w, x, ids):
    h, n = x.double(), x.shape[0]
    pos = torch.arange(n, device=DEV)
    bias = w["rel_bias"].double()[_bucket(pos[None, :] - pos[:, None])].permute(2, 0, 1)
    bias = bias.masked_fill(torch.from_numpy(ids == 0).to(DEV)[None, None, :], -math.inf)
    for i in range(2):
        p = "blk.%d." % i
        lin = lambda a, name: a @ w[p + name].double().T  # noqa: B023
        a = _rms(h, w[p + "attn_norm"].double(), 1e-6)
        q, k, v = (lin(a, c).reshape(n, 32, 64).transpose(0, 1).contiguous() for c in "qkv")
        h = h + lin(_attend(q, k, v, 1.0, bias).transpose(0, 1).reshape(n, 2048), "o")
        a = _rms(h, w[p + "ffn_norm"].double(), 1e-6)
        g = lin(a, "wi_0")
        g = 0.5 * g * (1 + torch.tanh(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3)))
        h = h + lin(g * lin(a, "wi_1"), "wo")
    return _rms(h, w["out_norm"].double(), 1e-6)


class _Dit64:
    """what the two transformers share, in 64 bits"""

    def __init__(self, w):
        self.w = w

    def lin(self, name, x):
        y = x @ self.w[name + ".weight"].double().T
        return y + self.w[name + ".bias"].double() if name + ".bias" in self.w else y

    def conv(self, name, x, pad):
        y = _conv(x, self.w[name + ".weight"], pad)
        return y + self.w[name + ".bias"].double() if name + ".bias" in self.w else y

    def swiglu(self, name, x):
        return _swiglu(x, *(self.w[name + c] for c in (".w1.weight", ".w3.weight", ".w2.weight")))

    def time(self, t, period):
        """the sinusoid arguments as the host computes them, in 32 bits"""
        k = np.arange(512, dtype=np.float32)
        f = (np.float32(10000.0 / period) * np.power(10000.0, (-2 * k / 1024).astype(np.float64)).astype(np.float32)).astype(np.float32)
        a = torch.from_numpy((t[:, None] * f[None, :]).astype(np.float64)).to(DEV)
        return self.lin("t_embed.mlp.2", _silu(self.lin("t_embed.mlp.0", torch.cat([torch.cos(a), torch.sin(a)], -1))))

    def attention(self, streams, last):
        """streams: [prefix, x, conditioning (B, S or 1, H), angles]; every stream's new x"""
        B, qs, ks, vs, ch = streams[0][1].shape[0], [], [], [], []
        for p, x, c, ang in streams:
            ch.append(self.lin(p + ".adaLN_modulation.1", c).chunk(2 if last and p != streams[0][0] else 6, -1))
            z = self.lin(p + ".attn.qkv", _ln(x) * (1 + ch[-1][1]) + ch[-1][0]).reshape(B, -1, 16, 64, 3)
            q = _rms(z[..., 0], self.w[p + ".attn.q_norm.weight"].double(), 1e-6)
            k = _rms(z[..., 1], self.w[p + ".attn.k_norm.weight"].double(), 1e-6)
            qs.append(q if ang is None else _rope(q, ang))
            ks.append(k if ang is None else _rope(k, ang))
            vs.append(z[..., 2])
        q, k, v = (torch.cat(a, 1).permute(0, 2, 1, 3).contiguous() for a in (qs, ks, vs))
        o = _attend(q, k, v, 0.125).permute(0, 2, 1, 3).reshape(B, -1, 1024)
        return ch, o.split([s[1].shape[1] for s in streams], 1)

    def block(self, streams, last=False):
        ch, o = self.attention(streams, last)
        out = []
        for i, (p, x, _, _) in enumerate(streams):
            if len(ch[i]) == 6:
                l1 = self.conv(p + ".linear1", o[i], 1) if self.w[p + ".linear1.weight"].dim() == 3 else self.lin(p + ".linear1", o[i])
                x = x + l1 * ch[i][2]
                r = _ln(x) * (1 + ch[i][4]) + ch[i][3]
                if p + ".ffn.fc1.weight" in self.w:
                    g = self.lin(p + ".ffn.fc1", r)
                    g = 0.5 * g * (1 + torch.tanh(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3)))
                    x = x + self.lin(p + ".ffn.fc2", g) * ch[i][5]
                else:
                    x = x + self.swiglu(p + ".ffn", r) * ch[i][5]
            out.append(x)
        return out

    def final(self, x, c):
        sh, sc = self.lin("final_layer.adaLN_modulation.1", c).chunk(2, -1)
        return _ln(x) * (1 + sc) + sh


def _exact_dit(m, w, s):
    n = _Dit64(w)
    c = _silu(n.time(s["t"], m.cfg.t_max_period))[:, None]
    lat, txt = n.lin("audio_input_proj", s["latent"].double().transpose(1, 2)), s["text"].double()
    ang = _angles(lat.shape[1])
    for i in range(7):
        p = "joint_blocks.%d." % i
        lat, txt = n.block([(p + "latent_block", lat, c, ang), (p + "text_block", txt, c, None)], last=i == 6)
    for i in range(14):
        lat, = n.block([("fused_blocks.%d" % i, lat, c, ang)])
    return n.lin("final_layer.linear", n.final(lat, c))


def _exact_graph(m, w, s):
    n = _Dit64(w)
    d = {k: v.double() for k, v in s.items() if k != "t"}
    lat = n.swiglu("audio_input_proj.2", _silu(n.conv("audio_input_proj.0", d["latent"].transpose(1, 2), 1)))
    clip = n.swiglu("clip_input_proj.2", _silu(n.lin("clip_input_proj.0", d["clip"])))
    T, Sc, Ss = lat.shape[1], clip.shape[1], d["sync"].shape[1]
    sync = d["sync"] + w["sync_pos_emb"].double()[torch.arange(Ss, device=DEV) % 8]
    sync = n.swiglu("sync_input_proj.2", _silu(n.conv("sync_input_proj.0", sync, 3)))
    txt = torch.cat([torch.nn.functional.pad(d["text"], (0, 1024)), d["t5"]], 1)
    txt = n.swiglu("text_input_proj.2", _silu(n.lin("text_input_proj.0", txt)))
    g = n.swiglu("global_cond_mlp", n.lin("clip_cond_proj", clip.mean(1)) + n.lin("text_cond_proj", d["g"]))
    g = (g + n.time(s["t"], m.cfg.t_max_period))[:, None]
    at = ((2 * torch.arange(T, device=DEV) + 1) * Ss).div(2 * T, rounding_mode="floor")
    c_lat, c = _silu(sync[:, at] + g), _silu(g)
    ang, ang_c = _angles(T), _angles(Sc, T / Sc)
    for i in range(2):
        p = "joint_blocks.%d." % i
        lat, clip, txt = n.block([(p + "latent_block", lat, c_lat, ang), (p + "clip_block", clip, c, ang_c),
                                  (p + "text_block", txt, c, None)], last=i == 1)
    lat, = n.block([("fused_blocks.0", lat, c_lat, ang)])
    return n.conv("final_layer.conv", n.final(lat, c_lat), 3)


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("t5", "vae", "dit", "graph"):
        return _exact_node(case, seed)
    m, w = _model(kind, case.get("type"))
    s = _model_inputs(case, seed)
    if kind == "t5":
        return _exact_t5(w, s["x"], s["ids"])
    if kind == "vae":
        return _exact_vae(w, s["latent"])
    return _exact_dit(m, w, s) if kind == "dit" else _exact_graph(m, w, s)
