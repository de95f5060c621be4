"""The work whose speed this library is held to, as a program on the C ABI has it done.

Everything a case needs is drawn on the GPU from a seed: quantized weights as blocks in device memory, bfloat16 weights as
host arrays (that is how they are uploaded), activations and tokens.  Results stay in device memory: a server samples
there, so logits and hidden rows are copied into the program's own tensors on the library's stream.

Kinds of work
  qmatmul     one quantized contraction, f32 in and out: the Linear of a program that keeps its own layers
  dequantize  a whole weight to f32: loading, merging, export
  prompt      a decoder takes a prompt in one pass; hidden rows of every token and the last token's logits come back
  decode      a decoder behind a prompt takes the next tokens one by one (sampling outside, so the tokens are given)
  request     a short prompt and the tokens behind it, from position 0: for models with recurrent layers, whose
              positions can only be fed in order

Decoder sizes are the layer shapes of bench.py, some with fewer layers (all layers of a model are alike, and the pass
through each is what is timed).
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from candy_amd import gulisun, hip, suvazen, synth

FORMATS = {"q4_0": synth.Q4_0, "q8_0": synth.Q8_0, "q4_k": synth.Q4_K, "q5_k": synth.Q5_K, "q6_k": synth.Q6_K}

# Layer shapes; Suvazen takes the first three as well (ffn: without the gate).
SIZES = {
    "8b": dict(d=4096, heads=32, kv=8, dim=128, ffn=14336, vocab=128256, down="q6_k", rope=500000.0),
    "7b": dict(d=4096, heads=32, kv=32, dim=128, ffn=11008, vocab=32000, down="q4_k", rope=10000.0),
    "1b": dict(d=2048, heads=32, kv=8, dim=64, ffn=8192, vocab=128256, down="q6_k", rope=500000.0),
}
# Gulisun: many small experts, few large ones.
MIXED = {
    "fine": dict(d=2048, vocab=102400, heads=16, dim=128, rot=64, vdim=128, kv_rank=512, q_rank=1024, lru=2560, blocks=10, taps=4,
                 experts=64, top=6, ff=1408, shared=2816),
    "coarse": dict(d=4096, vocab=32000, heads=32, dim=128, rot=64, vdim=128, kv_rank=512, q_rank=1536, lru=4096, blocks=16, taps=4,
                   experts=16, top=4, ff=2048, shared=6144),
}
SHAPES = ((4096, 4096), (1024, 4096), (11008, 4096), (4096, 11008), (14336, 4096), (4096, 14336), (32000, 4096), (8192, 2048),
          (2048, 8192), (3000, 2560))
EPS = 1e-5
WINDOW, CAP, LOGIT_CAP = 1536, 40.0, 25.0


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one token through a down projection: two launches and 25 MB, about the smallest call there is
        dict(name="matvec q4_k 4096x11008", kind="qmatmul", fmt="q4_k", rows=4096, cols=11008, m=1),
        # a handful of sequences, or drafted tokens, through a down projection
        dict(name="qmatmul q6_k 4096x14336 m6", kind="qmatmul", fmt="q6_k", rows=4096, cols=14336, m=6),
        # a short ragged prompt, or a batch of requests, through an up projection
        dict(name="qmatmul q8_0 11008x4096 m77", kind="qmatmul", fmt="q8_0", rows=11008, cols=4096, m=77),
        # a weight back to f32
        dict(name="dequantize q4_k 4096x11008", kind="dequantize", fmt="q4_k", rows=4096, cols=11008),
        # batch-1 generation behind a prompt, the usual 8B model with its f32 cache
        dict(name="llama 8b decode", kind="decode", model="llama", size="8b", layers=32, prompt=600, steps=4, f16=False),
        # a long context with the half-size cache
        dict(name="llama 7b decode long", kind="decode", model="llama", size="7b", layers=32, prompt=2000, steps=4, f16=True),
        # the prompt of a chat turn
        dict(name="llama 8b prompt 512", kind="prompt", model="llama", size="8b", layers=32, n=512, f16=False),
        # a longer, ragged prompt through a small model
        dict(name="llama 1b prompt 1500", kind="prompt", model="llama", size="1b", layers=16, n=1500, f16=False),
        # generation with bfloat16 weights, the window in use
        dict(name="suvazen 1b decode", kind="decode", model="suvazen", size="1b", layers=16, prompt=1700, steps=4, f16=False),
        # a document with bfloat16 weights, longer than the window
        dict(name="suvazen 8b prompt 2000", kind="prompt", model="suvazen", size="8b", layers=8, n=2000, f16=False),
        # a whole short request on the mixed model: prompt, then token by token
        dict(name="gulisun fine request", kind="request", model="gulisun", size="fine", layers=4, n=100, steps=16),
        # a long prompt over many experts
        dict(name="gulisun fine prompt 2048", kind="prompt", model="gulisun", size="fine", layers=4, n=2048, f16=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(("qmatmul", "qmatmul", "qmatmul", "dequantize", "llama", "llama", "suvazen", "suvazen", "gulisun", "gulisun"))
    if what in ("qmatmul", "dequantize"):
        rows, cols = rng.choice(SHAPES)
        rows -= rng.choice((0, 0, 0, rng.randrange(64)))
        case = dict(kind=what, fmt=rng.choice(sorted(FORMATS)), rows=rows, cols=cols)
        return case if what == "dequantize" else dict(case, m=_log_int(rng, 1, 1500))
    if what == "gulisun":
        size = rng.choice(sorted(MIXED))
        if rng.random() < 0.5:
            return dict(kind="request", model=what, size=size, layers=4, n=_log_int(rng, 2, 400), steps=rng.randint(2, 16))
        return dict(kind="prompt", model=what, size=size, layers=4, n=_log_int(rng, 16, 2048), f16=False)
    size, f16 = rng.choice(sorted(SIZES)), what == "llama" and rng.random() < 0.3
    layers = rng.randint(3, 8)
    if rng.random() < 0.5:
        return dict(kind="decode", model=what, size=size, layers=layers, prompt=_log_int(rng, 8, 2000), steps=rng.randint(1, 8), f16=f16)
    return dict(kind="prompt", model=what, size=size, layers=layers, n=_log_int(rng, 16, 2048), f16=f16)


# ------------------------------------------------------------------ the library
_device = None


class _Device(hip.Device):
    """Uploads bfloat16 weights from pinned memory, as a loader in a hurry does."""

    staging = None

    def dense(self, bits):
        n = bits.size
        if self.staging is None or self.staging.numel() < n:
            self.staging = None
            self.staging = torch.empty(n, dtype=torch.int16, pin_memory=True)
        staged = self.staging.numpy()[:n].view(np.uint16).reshape(bits.shape)
        np.copyto(staged, bits)
        return super().dense(staged)


def _dev():
    global _device
    if _device is None:
        _device = _Device(0)
    return _device


def _call(status):
    if status:
        raise RuntimeError(hip.lib().candy_hip_last_error().decode(errors="replace"))


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


# ------------------------------------------------------------------ quantized weights
# Levels bunch around the middle as those of a quantized normal distribution do.
_BELL = (1, 3, 4, 5, 5, 6, 7, 7, 8, 8, 9, 10, 10, 11, 12, 14)


def _bytes(n, count, g):
    return torch.randint(0, 256, (n, count), dtype=torch.uint8, device="cuda", generator=g)


def _bell_nibbles(n, count, g):
    table = torch.tensor([_BELL[b & 15] | _BELL[b >> 4] << 4 for b in range(256)], dtype=torch.uint8, device="cuda")
    out = _bytes(n, count, g)
    for part in out.split(1 << 17):  # index tensors are eight times as wide
        part.copy_(table[part.int()])
    return out


def _spread(n, g, scale):
    """fp16 block scales around `scale`, as bytes."""
    d = (torch.rand(n, 1, device="cuda", generator=g) * 0.6 + 0.7) * scale
    return d.half()


def _six_bit(n, g):
    """Packed 6-bit scales and minima of eight sub-blocks, the minima near the scales."""
    sc = torch.randint(33, 63, (n, 8), device="cuda", generator=g, dtype=torch.int32)
    mn = sc + torch.randint(-1, 2, (n, 8), device="cuda", generator=g, dtype=torch.int32)
    a, b, p, q = sc[:, :4], sc[:, 4:], mn[:, :4], mn[:, 4:]
    return torch.cat([a | (b >> 4) << 6, p | (q >> 4) << 6, (b & 15) | (q & 15) << 4], 1).to(torch.uint8)


def _blocks(fmt, rows, cols, g, std):
    """Blocks of a [rows, cols] weight about `std` wide: uint8 [blocks, block bytes]."""
    n = rows * cols // synth.BLOCK_ELEMS[FORMATS[fmt]]
    if fmt == "q4_0":
        parts = [_spread(n, g, std / 3.4).view(torch.uint8), _bell_nibbles(n, 16, g)]
    elif fmt == "q8_0":
        q = (torch.randn(n, 32, device="cuda", generator=g) * 42).round_().clamp_(-127, 127).to(torch.int8)
        parts = [_spread(n, g, std / 42).view(torch.uint8), q.view(torch.uint8)]
    elif fmt == "q4_k":
        d = _spread(n, g, std / 161)
        parts = [d.view(torch.uint8), (d * 7.5).view(torch.uint8), _six_bit(n, g), _bell_nibbles(n, 128, g)]
    elif fmt == "q5_k":
        d = _spread(n, g, std / 440)
        parts = [d.view(torch.uint8), (d * 15.5).view(torch.uint8), _six_bit(n, g), _bytes(n, 160, g)]
    else:
        sc = torch.randint(20, 61, (n, 16), device="cuda", generator=g, dtype=torch.int16)
        sc = torch.where(torch.randint(0, 2, (n, 16), device="cuda", generator=g, dtype=torch.uint8) > 0, sc, -sc).to(torch.int8)
        parts = [_bytes(n, 192, g), sc.view(torch.uint8), _spread(n, g, std / 780).view(torch.uint8)]
    return torch.cat(parts, 1)


def _values(fmt, blocks, rows, cols):
    """Blocks -> float64 [rows, cols], from the formats' descriptions."""
    def half(lo):
        return blocks[:, lo:lo + 2].contiguous().view(torch.float16).double()

    def sub_scales(lo):
        s = blocks[:, lo:lo + 12].int()
        a, p, hi = s[:, :4], s[:, 4:8], s[:, 8:]
        sc = torch.cat([a & 63, (hi & 15) | (a >> 6) << 4], 1)
        mn = torch.cat([p & 63, (hi >> 4) | (p >> 6) << 4], 1)
        return sc.double(), mn.double()

    n = blocks.shape[0]
    if fmt == "q4_0":
        q = blocks[:, 2:]
        v = (torch.stack([q & 15, q >> 4], 2).reshape(n, 32).double() - 8) * half(0)
    elif fmt == "q8_0":
        v = blocks[:, 2:].contiguous().view(torch.int8).double() * half(0)
    elif fmt in ("q4_k", "q5_k"):
        sc, mn = sub_scales(4)
        qs = blocks[:, -128:].reshape(n, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
        if fmt == "q5_k":
            bit = torch.arange(8, device="cuda", dtype=torch.uint8)[None, :, None]
            q = q | ((blocks[:, 16:48].reshape(n, 1, 32) >> bit) & 1) << 4
        v = (half(0) * sc)[:, :, None] * q.double() - (half(2) * mn)[:, :, None]
    else:
        ql, qh = blocks[:, :128].reshape(n, 2, 2, 32), blocks[:, 128:192].reshape(n, 2, 32)
        level = [(ql[:, :, j & 1] >> (4 * (j >> 1)) & 15) | (qh >> (2 * j) & 3) << 4 for j in range(4)]
        q = torch.stack(level, 2).reshape(n, 16, 16).double() - 32
        v = (half(208) * blocks[:, 192:208].contiguous().view(torch.int8).double())[:, :, None] * q
    return v.reshape(rows, cols)


def _qtensor(fmt, rows, cols, blocks):
    """A weight around blocks in device memory (room for a wide load past the last block behind them)."""
    nbytes = blocks.numel()
    room = torch.empty(nbytes + 64, dtype=torch.uint8, device="cuda")
    room[:nbytes] = blocks.reshape(-1)
    room[nbytes:] = 0
    torch.cuda.synchronize()
    h = ctypes.c_void_p()
    _call(hip.lib().candy_hip_qtensor_wrap(_dev().handle, FORMATS[fmt], rows, cols, room.data_ptr(), nbytes + 64, ctypes.byref(h)))
    q = hip.QTensor.__new__(hip.QTensor)
    q.dev, q.fmt, q.rows, q.cols, q.nbytes, q.handle, q._blocks = _dev(), FORMATS[fmt], rows, cols, nbytes, h.value, room
    return q


# ------------------------------------------------------------------ decoders
def _llama_matrices(case):
    """(kind, layer, format, rows, cols, std): projections into the residual stream are the narrower the more there are."""
    c = SIZES[case["size"]]
    d, qd, kd = c["d"], c["heads"] * c["dim"], c["kv"] * c["dim"]
    out = 0.01 / math.sqrt(2 * case["layers"])
    for l in range(case["layers"]):
        yield from ((hip.W_Q, l, "q4_k", qd, d, 0.02), (hip.W_K, l, "q4_k", kd, d, 0.02), (hip.W_V, l, "q4_k", kd, d, 0.02),
                    (hip.W_O, l, "q4_k", d, qd, out), (hip.W_GATE, l, "q4_k", c["ffn"], d, 0.02), (hip.W_UP, l, "q4_k", c["ffn"], d, 0.02),
                    (hip.W_DOWN, l, c["down"], d, c["ffn"], out))
    yield hip.W_HEAD, -1, "q6_k", c["vocab"], d, 0.02
    yield hip.W_EMBED, -1, "q8_0", c["vocab"], d, 1.5


def _matrix_gen(seed, kind, layer):
    return _gen(seed * 1000003 + (layer + 1) * 16 + kind)


def _norm_weight(seed, what, n):
    """Host f32 norm weight."""
    rng = np.random.Generator(np.random.Philox([seed, what]))
    return (1 + 0.1 * rng.standard_normal(n)).astype(np.float32)


def _positions(case):
    return case["n"] + case.get("steps", 0) if "n" in case else case["prompt"] + case["steps"]


def _tokens(case, seed):
    vocab = (MIXED if case["model"] == "gulisun" else SIZES)[case["size"]]["vocab"]
    return [int(t) for t in np.random.default_rng(seed).integers(0, vocab, _positions(case))]


def _build_llama(case, seed):
    c = SIZES[case["size"]]
    model = hip.Llama(_dev(), n_layers=case["layers"], d_model=c["d"], n_heads=c["heads"], n_kv_heads=c["kv"], head_dim=c["dim"],
                      d_ffn=c["ffn"], vocab=c["vocab"], max_pos=_positions(case) + 8, rms_eps=EPS, rope_base=c["rope"])
    for kind, l, fmt, rows, cols, std in _llama_matrices(case):
        model.set_qweight(kind, l, _qtensor(fmt, rows, cols, _blocks(fmt, rows, cols, _matrix_gen(seed, kind, l), std)))
    for l in range(case["layers"]):
        model.set_norm(hip.W_ATTN_NORM, l, _norm_weight(seed, 2 * l, c["d"]))
        model.set_norm(hip.W_FFN_NORM, l, _norm_weight(seed, 2 * l + 1, c["d"]))
    model.set_norm(hip.W_OUT_NORM, -1, _norm_weight(seed, 9999, c["d"]))
    if case["f16"]:
        model.set_kv_f16(True)
    return model


class _Pool:
    """bfloat16 matrices of a model cut from one run of normal values, each from its own place: a quick way to fill one."""

    N = 1 << 26

    def __init__(self, seed, std):
        self.run = (torch.randn(self.N, device="cuda", generator=_gen(seed)) * std).bfloat16()
        self.host = None

    def _at(self, name, count):
        return int.from_bytes(name.encode(), "little") % 1000003 * 64 % max(self.N - count, 1)

    def bits(self, name, shape):
        if self.host is None:
            self.host = self.run.view(torch.int16).cpu().numpy().view(np.uint16)
        count = math.prod(shape)
        lo = self._at(name, count)
        flat = self.host[lo:lo + count] if lo + count <= self.N else np.resize(self.host, count)
        return flat.reshape(shape)

    def values(self, name, shape):
        """The same as float64 on the GPU."""
        count = math.prod(shape)
        lo = self._at(name, count)
        flat = self.run[lo:lo + count] if lo + count <= self.N else self.run.repeat(-(-count // self.N))[:count]
        return flat.double().reshape(shape)


class _Weights:
    """The tensors of a bfloat16 model by name, as its loader asks for them."""

    def __init__(self, seed, shapes):
        self.seed, self.shape, self.pool = seed, shapes, _Pool(seed, 0.025)

    def __contains__(self, name):
        return True

    def bits(self, name):
        return self.pool.bits(name, self.shape(name))

    def f32(self, name):
        rng = np.random.Generator(np.random.Philox([self.seed, int.from_bytes(name.encode(), "little") % 1000003]))
        x = rng.standard_normal(self.shape(name)).astype(np.float32)
        if "norm" in name.rsplit(".", 1)[-1]:
            return (0.7 + 0.1 * x).astype(np.float32)
        if name.endswith("lam"):   # decays of a state that remembers tens to hundreds of tokens
            return (-4.5 + 0.7 * x).astype(np.float32)
        if name.endswith("conv"):
            return (0.5 * x).astype(np.float32)
        return (0.05 * x).astype(np.float32)

    def matrix(self, name):
        return self.pool.values(name, self.shape(name))

    def vector(self, name):
        return torch.from_numpy(self.f32(name)).cuda().double()


def _suvazen_config(case):
    c = SIZES[case["size"]]
    mixer = {"heads": c["heads"], "kv_heads": c["kv"], "dim": c["dim"], "scale": c["dim"] ** -0.5, "softcap": CAP, "mask": {"size": WINDOW},
             "rot": {"base": 500000.0, "dims": c["dim"] // 2, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}
    return {"vocab": c["vocab"], "width": c["d"], "norm": {"eps": EPS}, "residual_mult": 0.5, "logit_scale": 1.0, "logit_softcap": LOGIT_CAP,
            "layers": [{"type": "attention", "mixer": mixer, "mlp": {"kind": "dense", "ff": c["ffn"]}} for _ in range(case["layers"])]}


def _suvazen_weights(case, seed):
    c = SIZES[case["size"]]
    qd, kd, d, ff = c["heads"] * c["dim"], c["kv"] * c["dim"], c["d"], c["ffn"]
    shapes = {"q": (qd, d), "k": (kd, d), "o": (d, qd), "up": (ff, d), "down": (d, ff), "embed": (c["vocab"], d), "head": (c["vocab"], d),
              "sink": (c["heads"],)}
    return _Weights(seed, lambda name: shapes.get(name.rsplit(".", 1)[-1], (d,)))


def _gulisun_config(case):
    """Of four layers, the first has a cache of its own, the second is recurrent, the third reads the first's cache, the
    fourth has its own and no sink."""
    c = MIXED[case["size"]]
    mlp = {"kind": "moe", "router": {"experts": c["experts"], "top": c["top"]}, "expert": {"ff": c["ff"]}, "shared": {"ff": c["shared"]}}
    layers = []
    for i in range(case["layers"]):
        kind = ("latent_attention", "rglru", "latent_attention", "latent_attention_2")[i % 4]
        mixer = {"heads": c["heads"], "dim": c["dim"], "rot_dim": c["rot"], "vdim": c["vdim"], "kv_rank": c["kv_rank"], "q_rank": c["q_rank"],
                 "scale": (c["dim"] + c["rot"]) ** -0.5, "rot": {"base": 500000.0, "dims": c["rot"]}}
        if kind == "rglru":
            mixer = {"width": c["lru"], "blocks": c["blocks"], "conv": c["taps"]}
        elif i % 4 == 2:
            mixer["kv_from"] = i - 2
        layers.append({"type": kind, "mixer": mixer, "mlp": mlp})
    return {"vocab": c["vocab"], "width": c["d"], "norm": {"eps": EPS}, "embedding": {"scale": 36.0}, "layers": layers}


def _gulisun_weights(case, seed):
    c, cfg = MIXED[case["size"]], _gulisun_config(case)
    d, H, size, u = c["d"], c["heads"], c["lru"] // c["blocks"], c["lru"]
    shapes = {"embed": (c["vocab"], d), "dq": (c["q_rank"], d), "uq": (H * (c["dim"] + c["rot"]), c["q_rank"]),
              "dkv": (c["kv_rank"] + c["rot"], d), "uk": (H * c["dim"], c["kv_rank"]), "uv": (H * c["vdim"], c["kv_rank"]), "y": (u, d),
              "x": (u, d), "ra": (c["blocks"], size, size), "ri": (c["blocks"], size, size), "router": (c["experts"], d),
              "dq.norm": (c["q_rank"],), "dkv.norm": (c["kv_rank"],), "sink": (H,), "conv": (u, c["taps"]), "y.b": (u,), "x.b": (u,),
              "conv.b": (u,), "ra.b": (u,), "ri.b": (u,), "lam": (u,), "norm1": (d,), "norm2": (d,), "final.norm": (d,)}

    def shape(name):
        if not name.startswith("l"):
            return shapes[name]
        layer, rest = name.split(".", 1)
        last = rest.split(".", 1)[-1]
        if last == "o":
            return (d, u) if cfg["layers"][int(layer[1:])]["type"] == "rglru" else (d, H * c["vdim"])
        if last in shapes:
            return shapes[last]
        ff = c["shared"] if "shared" in last else c["ff"]
        return (ff, d) if last.endswith("up") else (d, ff)

    return _Weights(seed, shape)


def _build(case, seed):
    room = _positions(case) + 8
    if case["model"] == "llama":
        return _build_llama(case, seed)
    if case["model"] == "suvazen":
        return suvazen.build(_dev(), _suvazen_config(case), _suvazen_weights(case, seed), room)
    return gulisun.build(_dev(), _gulisun_config(case), _gulisun_weights(case, seed), room)


# ------------------------------------------------------------------ a pass
def prepare(case, seed):
    torch.cuda.synchronize()
    g = _gen(seed)
    state = {"case": case}
    if case["kind"] in ("qmatmul", "dequantize"):
        rows, cols, m = case["rows"], case["cols"], case.get("m", case["rows"])
        state["w"] = _qtensor(case["fmt"], rows, cols, _blocks(case["fmt"], rows, cols, g, 0.02))
        if case["kind"] == "qmatmul":
            state["x"] = torch.randn(m, cols, device="cuda", generator=g)
        state["y"] = torch.empty(m, rows if case["kind"] == "qmatmul" else cols, device="cuda")
        torch.cuda.synchronize()
        return state
    model, tokens = _build(case, seed), _tokens(case, seed)
    state["model"] = model
    state["ids"] = (ctypes.c_int32 * len(tokens))(*tokens)
    steps = case.get("steps", 1)
    state["logits"] = torch.empty(steps + (case["kind"] == "request"), model.vocab, device="cuda")
    if case["kind"] == "decode":
        model.prefill(tokens[:case["prompt"]], 0, want_logits=False)
    else:
        state["hidden"] = torch.empty(case["n"], model.width, device="cuda")
    torch.cuda.synchronize()
    return state


def _prefill(s, n, logits):
    """A prompt; its last token's logits and every token's hidden row into the program's tensors."""
    L, dev, model = hip.lib(), s["model"].dev.handle, s["model"]
    lg, rows, ld = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_int64()
    _call(L.candy_hip_decoder_prefill(model.handle, s["ids"], n, 0, ctypes.byref(lg), None))
    _call(L.candy_hip_d2d(dev, logits.data_ptr(), lg, 4 * model.vocab))
    _call(L.candy_hip_decoder_prompt_hidden(model.handle, ctypes.byref(rows), ctypes.byref(ld)))
    _call(L.candy_hip_d2d(dev, s["hidden"].data_ptr(), rows, 4 * n * ld.value))  # every width here is unpadded


def _decode(s, pos, logits):
    L, dev, model = hip.lib(), s["model"].dev.handle, s["model"]
    lg = ctypes.c_void_p()
    for k in range(logits.shape[0]):
        _call(L.candy_hip_decoder_decode(model.handle, s["ids"][pos + k], pos + k, ctypes.byref(lg), None))
        _call(L.candy_hip_d2d(dev, logits[k].data_ptr(), lg, 4 * model.vocab))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "qmatmul":
        _call(hip.lib().candy_hip_qmatmul(_device.handle, state["w"].handle, state["x"].data_ptr(), case["m"], state["y"].data_ptr()))
        return state["y"]
    if kind == "dequantize":
        _call(hip.lib().candy_hip_dequantize(_device.handle, state["w"].handle, state["y"].data_ptr()))
        return state["y"]
    if kind == "decode":
        _decode(state, case["prompt"], state["logits"])
        return {"logits": state["logits"]}
    _prefill(state, case["n"], state["logits"][0])
    if kind == "request":
        _decode(state, case["n"], state["logits"][1:])
    return {"logits": state["logits"], "hidden": state["hidden"]}


# ------------------------------------------------------------------ what a pass cannot do without
def _layer_work(case):
    """Per layer, averaged over the layers: weight values by (bytes each), multiply-adds per token in projections, head
    dims of attention (per query and key), cache bytes per position."""
    if case["model"] == "gulisun":
        c = MIXED[case["size"]]
        d, H, dk = c["d"], c["heads"], c["dim"] + c["rot"]
        shared = 2 * d * c["shared"] + d * c["experts"]
        expert = 2 * d * c["ff"]
        attn = d * c["q_rank"] + H * dk * c["q_rank"] + H * (c["dim"] + c["vdim"]) * c["kv_rank"] + d * H * c["vdim"]
        down = d * (c["kv_rank"] + c["rot"])
        lru = c["lru"] * (3 * d + 2 * c["lru"] // c["blocks"])
        mixers = (3 * attn + 2 * down + lru) / 4
        return dict(weights=2 * (mixers + shared), expert=2 * expert, experts=c["experts"], top=c["top"],
                    macs=mixers + shared + c["top"] * expert, attn=0.75 * H * (dk + c["vdim"]), cache=0.75 * 2 * (c["kv_rank"] + c["rot"]))
    c = SIZES[case["size"]]
    d, qd, kd, ff = c["d"], c["heads"] * c["dim"], c["kv"] * c["dim"], c["ffn"]
    if case["model"] == "suvazen":
        values = d * (qd + kd) + d * qd + 2 * d * ff
        return dict(weights=2 * values, expert=0, experts=0, top=0, macs=values, attn=2 * qd, cache=4 * kd)
    values = d * (2 * qd + 2 * kd + 2 * ff)
    weights = values * 144 / 256 + d * ff * (210 if c["down"] == "q6_k" else 144) / 256
    return dict(weights=weights, expert=0, experts=0, top=0, macs=values + d * ff, attn=2 * qd, cache=2 * kd * (2 if case["f16"] else 4))


def _model_work(case, n, pos0):
    """n tokens at once behind pos0 others, logits of the last one."""
    w, L = _layer_work(case), case["layers"]
    c = (MIXED if case["model"] == "gulisun" else SIZES)[case["size"]]
    window = WINDOW if case["model"] == "suvazen" else 1 << 30
    pairs = sum(min(p + 1, window) for p in range(pos0, pos0 + n))
    seen = min(pos0, window) if n == 1 else min(pos0, window + n)
    head = c["vocab"] * c["d"]
    touched = min(w["experts"], n * w["top"])
    nbytes = L * (w["weights"] + touched * w["expert"] + w["cache"] * (seen + n)) + head * (210 / 256 if case["model"] == "llama" else 2) + \
        4 * c["vocab"]
    flops = 2 * (L * (n * w["macs"] + pairs * w["attn"]) + head)
    return nbytes, flops


def work(case):
    if case["kind"] in ("qmatmul", "dequantize"):
        f = FORMATS[case["fmt"]]
        rows, cols = case["rows"], case["cols"]
        weight = rows * cols // synth.BLOCK_ELEMS[f] * synth.BLOCK_BYTES[f]
        if case["kind"] == "dequantize":
            return {"bytes": weight + 4 * rows * cols, "flops": rows * cols}
        return {"bytes": weight + 4 * case["m"] * (rows + cols), "flops": 2 * case["m"] * rows * cols}
    c = (MIXED if case["model"] == "gulisun" else SIZES)[case["size"]]
    nbytes = flops = 0
    if "n" in case:
        nbytes, flops = _model_work(case, case["n"], 0)
        nbytes += 4 * case["n"] * c["d"]
    for k in range(case.get("steps", 0)):
        b, f = _model_work(case, 1, (case["n"] if "n" in case else case["prompt"]) + k)
        nbytes, flops = nbytes + b, flops + f
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the distance from 64 bits.  A contraction of few rows is exact but for f32 sums; more rows round both
    operands to fp16 once.  A quantized decoder re-quantizes its activations in front of every projection, so that a
    last-place difference moves some levels (1/127 of a block's range each); bfloat16 decoders round theirs.  Expert choices
    tip over at near ties, which moves whole rows."""
    if case["kind"] == "dequantize":
        return "exact"
    if case["kind"] == "qmatmul":
        tiles = case["m"] >= (33 if case["fmt"] in ("q4_k", "q6_k") else 65)
        return {"rel": 1.2e-3 if tiles else 1e-5}
    return {"rel": 0.016 if case["model"] == "suvazen" else 0.03, "max": 0.9}


# ------------------------------------------------------------------ the same in 64 bits
def _q8(x):
    """Activations as the quantizer of the contraction leaves them: per 32 values, levels of amax / 127 in f32."""
    b = x.float().reshape(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127
    q = torch.where(d > 0, b / d, torch.zeros_like(b)).double()
    q = torch.sign(q) * torch.floor(q.abs() + 0.5)
    return (q * d.half().double()).reshape(x.shape)


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _layer_norm(x, w, b):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w + b


def _turn(x, freq):
    """Pairs (i, i + dims/2) of the first dims values of [tokens, heads, dim], dims = 2 len(freq)."""
    half = len(freq)
    ang = torch.arange(x.shape[0], device="cuda", dtype=torch.float64)[:, None, None] * torch.tensor(freq, device="cuda", dtype=torch.float64)
    u, v = x[..., :half], x[..., half:2 * half]
    return torch.cat([u * ang.cos() - v * ang.sin(), v * ang.cos() + u * ang.sin(), x[..., 2 * half:]], -1)


def _frequencies(base, dims):
    return [base ** (-2.0 * i / dims) for i in range(dims // 2)]


def _attend(q, k, v, scale, cap=None, window=None, sink=None):
    """q, k, v [tokens, heads, dim], causal; fewer heads of k and v are shared by neighbouring heads of q."""
    n, H = q.shape[0], q.shape[1]
    pos = torch.arange(n, device="cuda")
    gap = pos[:, None] - pos[None, :]
    hidden = (gap < 0) | (gap >= (window or n))
    out = []
    for h in range(H):
        g = h * k.shape[1] // H
        s = q[:, h] @ k[:, g].T * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        s = s.masked_fill(hidden, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].expand(n, 1)], 1)
        out.append(torch.softmax(s, 1)[:, :n] @ v[:, g])
    return torch.stack(out, 1).reshape(n, -1)


def _exact_llama(case, seed, tokens):
    c = SIZES[case["size"]]
    at = {(kind, l): (fmt, rows, cols, std) for kind, l, fmt, rows, cols, std in _llama_matrices(case)}

    def matrix(kind, l):
        fmt, rows, cols, std = at[kind, l]
        return fmt, _blocks(fmt, rows, cols, _matrix_gen(seed, kind, l), std), rows, cols

    def linear(kind, l, xq):
        return xq @ _values(*matrix(kind, l)).T

    def norm(what):
        return torch.from_numpy(_norm_weight(seed, what, c["d"])).cuda().double()

    fmt, blocks, rows, cols = matrix(hip.W_EMBED, -1)
    picked = blocks.reshape(rows, -1)[torch.tensor(tokens, device="cuda")]
    x = _values(fmt, picked.reshape(-1, blocks.shape[1]), len(tokens), cols)
    freq, n = _frequencies(c["rope"], c["dim"]), len(tokens)
    for l in range(case["layers"]):
        a = _q8(_rms(x, norm(2 * l)))
        q, k, v = (linear(kind, l, a).reshape(n, -1, c["dim"]) for kind in (hip.W_Q, hip.W_K, hip.W_V))
        q, k = _turn(q, freq), _turn(k, freq)
        if case["f16"]:
            k, v = k.half().double(), v.half().double()
        x = x + linear(hip.W_O, l, _q8(_attend(q, k, v, c["dim"] ** -0.5)))
        a = _q8(_rms(x, norm(2 * l + 1)))
        x = x + linear(hip.W_DOWN, l, _q8(torch.nn.functional.silu(linear(hip.W_GATE, l, a)) * linear(hip.W_UP, l, a)))
    return x, lambda rows_: linear(hip.W_HEAD, -1, _q8(_rms(rows_, norm(9999))))


def _exact_suvazen(case, seed, tokens):
    c, w, n = SIZES[case["size"]], _suvazen_weights(case, seed), len(tokens)
    freq = []
    for f in _frequencies(500000.0, c["dim"] // 2):
        wave = 2 * math.pi / f
        if wave > 8192 / 1.0:
            f /= 8.0
        elif wave >= 8192 / 4.0:
            mix = (8192 / wave - 1.0) / (4.0 - 1.0)
            f = (1 - mix) * f / 8.0 + mix * f
        freq.append(f)

    def norm(name, x):
        return _layer_norm(x, w.vector(name), w.vector(name + ".b"))

    x = w.matrix("embed")[torch.tensor(tokens, device="cuda")]
    for l in range(case["layers"]):
        p = "l%d" % l
        a = norm(p + ".norm1", x)
        q, k = ((a @ w.matrix(p + ".mix." + m).T).reshape(n, -1, c["dim"]) for m in "qk")
        a = _attend(_turn(q, freq), _turn(k, freq), k, c["dim"] ** -0.5, CAP, WINDOW, w.vector(p + ".mix.sink"))
        x = x + 0.5 * norm(p + ".norm1b", a @ w.matrix(p + ".mix.o").T)
        a = torch.relu(norm(p + ".norm2", x) @ w.matrix(p + ".mlp.up").T)
        x = x + 0.5 * norm(p + ".norm2b", (a * a) @ w.matrix(p + ".mlp.down").T)
    return x, lambda rows: LOGIT_CAP * torch.tanh(norm("final.norm", rows) @ w.matrix("head").T / LOGIT_CAP)


def _exact_gulisun(case, seed, tokens):
    c, w, n = MIXED[case["size"]], _gulisun_weights(case, seed), len(tokens)
    H, freq, latents = c["heads"], _frequencies(500000.0, c["rot"]), {}

    def latent_attention(x, l, source, sink):
        p = "l%d.mix." % l
        if source == l:
            z = x @ w.matrix(p + "dkv").T
            latents[l] = _rms(z[:, :c["kv_rank"]], w.vector(p + "dkv.norm")), _turn(z[:, None, c["kv_rank"]:], freq)
        lat, turned = latents[source]
        q = (_rms(x @ w.matrix(p + "dq").T, w.vector(p + "dq.norm")) @ w.matrix(p + "uq").T).reshape(n, H, -1)
        q = torch.cat([q[..., :c["dim"]], _turn(q[..., c["dim"]:].contiguous(), freq)], -1)
        k = torch.cat([(lat @ w.matrix(p + "uk").T).reshape(n, H, -1), turned.expand(n, H, -1)], -1)
        v = (lat @ w.matrix(p + "uv").T).reshape(n, H, -1)
        a = _attend(q, k, v, (c["dim"] + c["rot"]) ** -0.5, sink=w.vector(p + "sink") if sink else None)
        return a @ w.matrix(p + "o").T

    def recurrent(x, l):
        p = "l%d.mix." % l
        y = torch.nn.functional.gelu(x @ w.matrix(p + "y").T + w.vector(p + "y.b"), approximate="tanh")
        v = x @ w.matrix(p + "x").T + w.vector(p + "x.b")
        taps, padded = w.vector(p + "conv"), torch.cat([torch.zeros(c["taps"] - 1, c["lru"], device="cuda", dtype=torch.float64), v])
        u = sum(padded[j:j + n] * taps[:, j] for j in range(c["taps"])) + w.vector(p + "conv.b")

        def gate(m):
            parts = u.reshape(n, c["blocks"], -1)
            g = w.matrix(p + m)
            return torch.sigmoid(torch.cat([parts[:, i] @ g[i].T for i in range(c["blocks"])], 1) + w.vector(p + m + ".b"))

        log_a = -8 * gate("ra") * torch.nn.functional.softplus(w.vector(p + "lam"))
        a, b = log_a.exp(), torch.sqrt(-torch.expm1(2 * log_a)) * gate("ri") * u
        s, out = torch.zeros(c["lru"], device="cuda", dtype=torch.float64), torch.empty_like(a)
        for t in range(n):
            s = a[t] * s + b[t]
            out[t] = s
        return (out * y) @ w.matrix(p + "o").T

    def experts(x, l):
        p = "l%d.mlp." % l

        def ff(h, name):
            h = torch.relu(h @ w.matrix(p + name + ".up").T)
            return (h * h) @ w.matrix(p + name + ".down").T

        weights, ids = torch.softmax(x @ w.matrix(p + "router").T, 1).topk(c["top"], 1)
        weights = weights / (weights.sum(1, keepdim=True) + 1e-20)
        out = ff(x, "shared")
        for e in range(c["experts"]):
            t, k = (ids == e).nonzero(as_tuple=True)
            if len(t):
                out[t] += weights[t, k][:, None] * ff(x[t], "e%d" % e)
        return out

    x = w.matrix("embed")[torch.tensor(tokens, device="cuda")] * 36.0
    for l in range(case["layers"]):
        y = recurrent(x, l) if l % 4 == 1 else latent_attention(x, l, l - 2 if l % 4 == 2 else l, l % 4 != 3)
        x = x + _rms(y, w.vector("l%d.norm1" % l))
        x = x + _rms(experts(x, l), w.vector("l%d.norm2" % l))
    return x, lambda rows: _rms(rows, w.vector("final.norm")) @ w.matrix("embed").T


def exact(case, seed):
    if case["kind"] in ("qmatmul", "dequantize"):
        g = _gen(seed)
        w = _values(case["fmt"], _blocks(case["fmt"], case["rows"], case["cols"], g, 0.02), case["rows"], case["cols"])
        if case["kind"] == "dequantize":
            return w
        return _q8(torch.randn(case["m"], case["cols"], device="cuda", generator=g)) @ w.T
    forward = {"llama": _exact_llama, "suvazen": _exact_suvazen, "gulisun": _exact_gulisun}[case["model"]]
    hidden, head = forward(case, seed, _tokens(case, seed))
    if case["kind"] == "decode":
        return {"logits": head(hidden[case["prompt"]:])}
    return {"logits": head(hidden[case["n"] - 1:]), "hidden": hidden[:case["n"]]}
