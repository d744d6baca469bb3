"""Timed workloads of the decode engine, as a program over its C ABI runs them.

Every case calls the public entry points through ``pycitlali`` on device
memory the caller owns (torch tensors).  Single operations are launched one by
one; a decoder layer and a whole decode step are captured once in a HIP graph
on the library's stream and replayed, the way ``QwenModel::decode_greedy``
runs them.  Weights are random K-quant blocks (or fp16 rows) whose values have
the spread and zero mean of trained ones; activations are normal with a few
large channels, as hidden states have.

Kinds of case:

* ``matvec``   one GEMV, Q4_K / Q6_K / fp16 weights, fp16 or fp32 output;
* ``head``     final norm + output projection, fp32 logits;
* ``attention``  one sequence's decode attention over its cache;
* ``batch``    many sequences of unequal length in one attention launch;
* ``load``     load-time dequantisation of a Q4_K and a Q6_K tensor to fp16;
* ``layer``    one decoder layer of a decode step, fused where the engine has
  a fused launch for the shape and launch by launch where it has not;
* ``model``    a whole decode step: embedding, layers, logits, greedy pick.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "citlali-llm-engine_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import pycitlali as hip  # noqa: E402
from pycitlali import device as dev  # noqa: E402

EPS = 1e-6
THETA = 1e6
BLOCK_BYTES = {"q4k": 144, "q6k": 210, "fp16": 512}   # per 256 weights
# weight types of one layer: Q4_K with Q6_K attn_v and ffn_down, all Q6_K, or all fp16
MIXES = {
    "q4km": dict(q="q4k", k="q4k", v="q6k", o="q4k", gate="q4k", up="q4k", down="q6k"),
    "q6k": dict.fromkeys(("q", "k", "v", "o", "gate", "up", "down"), "q6k"),
    "fp16": dict.fromkeys(("q", "k", "v", "o", "gate", "up", "down"), "fp16"),
}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call a decode makes: one FFN projection of a 0.6B-class model, bound by its launch
        dict(name="matvec_q4k_small", kind="matvec", quant="q4k", rows=3072, cols=1024, f32=True),
        # one decode step's attention of a 0.6B-class model at a short context
        dict(name="attention_short", kind="attention", heads=16, kv_heads=8, head_dim=128, length=1024,
             max_context=1024),
        # a layer of an 8B-class model at a usual context: the main path of the engine
        dict(name="layer_8b", kind="layer", mix="q4km", hidden=4096, ffn=12288, heads=32, kv_heads=8, head_dim=128,
             length=8192, max_context=8192, bias=False, qk_norm=True),
        # a layer of a 14B-class model (row lengths that end in a partial wave step, 5 heads per kv head)
        dict(name="layer_14b", kind="layer", mix="q4km", hidden=5120, ffn=17408, heads=40, kv_heads=8, head_dim=128,
             length=2001, max_context=4096, bias=False, qk_norm=True),
        # a layer loaded as fp16 (DequantizeToFp16), 4B-class
        dict(name="layer_4b_fp16", kind="layer", mix="fp16", hidden=2560, ffn=9728, heads=32, kv_heads=8,
             head_dim=128, length=701, max_context=2048, bias=False, qk_norm=True),
        # a qwen2-style layer (biases, no head norms) of sizes outside the Qwen3 family: the unfused launches
        dict(name="layer_biased", kind="layer", mix="q4km", hidden=3584, ffn=18944, heads=28, kv_heads=4,
             head_dim=128, length=3001, max_context=4096, bias=True, qk_norm=False),
        # the output projection of an 8B-class model, the largest GEMV of a step
        dict(name="head_8b", kind="head", quant="q6k", rows=151936, cols=4096),
        # one long document: a single sequence's attention past 30k positions
        dict(name="attention_long", kind="attention", heads=32, kv_heads=8, head_dim=128, length=30011,
             max_context=32768),
        # serving: 16 long sequences decoded in one launch
        dict(name="batch_long", kind="batch", nseq=16, heads=32, kv_heads=8, head_dim=128, shortest=4096,
             longest=32768),
        # serving a head_dim-64 model: many chat-length sequences
        dict(name="batch_hd64", kind="batch", nseq=48, heads=32, kv_heads=4, head_dim=64, shortest=200,
             longest=6000),
        # loading a model as fp16: an FFN's Q4_K and Q6_K tensors dequantised on the device
        dict(name="load_ffn", kind="load", q4k=12288 * 4096, q6k=4096 * 12288),
        # a whole decode step of a 0.6B-class model: embedding to logits and greedy pick
        dict(name="model_0p6b", kind="model", mix="q4km", layers=28, hidden=1024, ffn=3072, heads=16, kv_heads=8,
             head_dim=128, vocab=151936, length=601, max_context=2048, bias=False, qk_norm=True),
    ]


def _logint(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _blocks(rng, lo, hi):
    """A row length: a multiple of 256, log-uniform."""
    return 256 * _logint(rng, lo // 256, hi // 256)


# hidden, ffn, heads, kv_heads of the model sizes the engine is run at
_SIZES = [(1024, 3072, 16, 8), (2048, 6144, 16, 8), (2560, 9728, 32, 8), (4096, 12288, 32, 8), (5120, 17408, 40, 8),
          (5120, 25600, 64, 8)]


def draw(rng):
    kind = rng.choice(("matvec", "matvec", "layer", "layer", "attention", "batch", "load", "head"))
    if kind == "matvec":
        quant = rng.choice(("q4k", "q6k", "fp16"))
        cols = rng.choice((1024, 2048, 2560, 4096, 5120, 9728, 12288, _blocks(rng, 256, 28672),
                           _blocks(rng, 256, 28672)))
        return dict(kind=kind, quant=quant, rows=_logint(rng, 200, (40 << 20) // cols), cols=cols,
                    f32=rng.random() < 0.3)
    if kind == "head":
        return dict(kind=kind, quant=rng.choice(("q4k", "q6k", "fp16")), rows=_logint(rng, 20000, 140000),
                    cols=rng.choice((1024, 2048, 2560, 4096)))
    if kind == "attention":
        kv = rng.choice((1, 2, 4, 8))
        group = rng.choice((1, 2, 3, 4, 5, 7, 8))
        length = _logint(rng, 32, 40000)
        return dict(kind=kind, heads=kv * group, kv_heads=kv, head_dim=rng.choice((64, 128, 128)), length=length,
                    max_context=length + rng.randrange(0, 4096))
    if kind == "batch":
        kv, group, hd = rng.choice((2, 4, 8)), rng.choice((1, 2, 4, 5, 7, 8)), rng.choice((64, 128, 128))
        longest = _logint(rng, 256, 32768)
        budget = 2.5e8 / (longest * kv * hd)
        return dict(kind=kind, nseq=_logint(rng, 2, max(2, min(128, int(budget)))), heads=kv * group, kv_heads=kv,
                    head_dim=hd, shortest=max(1, int(longest * rng.uniform(0.02, 0.9))), longest=longest)
    if kind == "load":
        return dict(kind=kind, q4k=_logint(rng, 100000, 60000000), q6k=_logint(rng, 100000, 60000000))
    length = _logint(rng, 64, 12000)
    if rng.random() < 0.6:
        hidden, ffn, heads, kv = rng.choice(_SIZES)
        return dict(kind=kind, mix=rng.choice(("q4km", "q4km", "q6k", "fp16")), hidden=hidden, ffn=ffn, heads=heads,
                    kv_heads=kv, head_dim=128, length=length, max_context=length + rng.randrange(1, 2048), bias=False,
                    qk_norm=True)
    hidden = _blocks(rng, 768, 6144)
    kv, group = rng.choice((2, 4, 8)), rng.choice((2, 4, 6, 7))
    return dict(kind=kind, mix=rng.choice(("q4km", "fp16")), hidden=hidden, ffn=_blocks(rng, 2048, 20480),
                heads=kv * group, kv_heads=kv, head_dim=128, length=length,
                max_context=length + rng.randrange(1, 2048), bias=rng.random() < 0.5, qk_norm=rng.random() < 0.5)


# ---------------------------------------------------------------- device data
class Buffer(dev.DeviceArray):
    """A torch tensor as a buffer argument of the bindings (torch owns it), in
    whole 4 KB pages as the library's own allocator hands memory out."""

    def __init__(self, tensor):
        n = tensor.numel() * tensor.element_size()
        if n % 4096:
            pages = torch.zeros(n + -n % 4096, dtype=torch.uint8, device=tensor.device)
            pages[:n].copy_(tensor.contiguous().view(-1).view(torch.uint8))
            tensor = pages[:n].view(tensor.dtype).view(tensor.shape)
        self.tensor = tensor
        self.ptr = tensor.data_ptr()
        self.nbytes = tensor.numel() * tensor.element_size()

    def close(self):
        self.ptr = 0


_stream = None


def _library():
    """The library on cuda:0, its launches on a stream of the program's own
    (graphs are captured and replayed there)."""
    global _stream
    if _stream is None:
        torch.cuda.init()
        hip.check(hip.load().citlali_hip_init(0))
        _stream = dev.Stream()
        dev.set_stream(_stream)


def _gen(seed):
    return torch.Generator("cuda").manual_seed(int(seed) * 7919 + 13)


def _half(*shape):
    return Buffer(torch.zeros(shape, dtype=torch.float16, device="cuda"))


def _normal(g, *shape, scale=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float16) * scale


def _hidden_state(g, n):
    """Normal values with about one channel in 200 twenty times larger."""
    big = (torch.rand(n, generator=g, device="cuda") < 0.005).half() * 19 + 1
    return _normal(g, n) * big


def _norm_weight(g, n):
    return (1 + 0.2 * torch.randn(n, generator=g, device="cuda")).half()


def _weight(g, quant, rows, cols, gain=1.0):
    """[rows][cols] of rms gain / sqrt(cols) and mean about 0."""
    if quant == "fp16":
        return _normal(g, rows, cols, scale=gain / math.sqrt(cols))
    n = rows * (cols // 256)
    b = torch.randint(0, 256, (n, BLOCK_BYTES[quant]), generator=g, device="cuda", dtype=torch.uint8)
    # rms of a random block's values: 258 d (Q4_K with dmin = 7.5 d), 1366 d (Q6_K)
    d = (0.5 + torch.rand(n, 1, generator=g, device="cuda")) * (gain / math.sqrt(cols))
    if quant == "q4k":
        d = d / 258
        b[:, 0:2] = d.half().view(torch.uint8)
        b[:, 2:4] = (7.5 * d).half().view(torch.uint8)
    else:
        b[:, 208:210] = (d / 1366).half().view(torch.uint8)
    return b


class Layer:
    """One decoder layer's weights and cache."""

    def __init__(self, g, c):
        h, f, nq, nkv = c["hidden"], c["ffn"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        self.types = MIXES[c["mix"]]
        self.shapes = dict(q=(nq, h), k=(nkv, h), v=(nkv, h), o=(h, nq), gate=(f, h), up=(f, h), down=(h, f))
        gains = dict(o=0.5, down=0.5)
        self.w = {n: Buffer(_weight(g, self.types[n], *self.shapes[n], gains.get(n, 1.0))) for n in self.shapes}
        self.bias = {n: Buffer(_normal(g, self.shapes[n][0], scale=0.1)) for n in ("q", "k", "v")} if c["bias"] else {}
        self.attn_norm, self.ffn_norm = Buffer(_norm_weight(g, h)), Buffer(_norm_weight(g, h))
        self.q_norm = self.k_norm = None
        if c["qk_norm"]:
            self.q_norm, self.k_norm = (Buffer(_norm_weight(g, c["head_dim"])) for _ in range(2))
        rows = (c["max_context"], c["kv_heads"], c["head_dim"])
        self.k_cache, self.v_cache = Buffer(_normal(g, *rows)), Buffer(_normal(g, *rows))


class Scratch:
    """The activations a decode step keeps."""

    def __init__(self, c):
        h, nq, nkv = c["hidden"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        self.x, self.x_alt, self.norm, self.proj, self.ffn_out = (_half(h) for _ in range(5))
        self.q, self.attn = _half(nq), _half(nq)
        self.k, self.v = _half(nkv), _half(nkv)
        self.gate, self.up, self.act = (_half(c["ffn"]) for _ in range(3))
        self.ws_bytes = dev.attention_workspace_bytes(c["max_context"], 1, c["heads"], c["kv_heads"], c["head_dim"])
        self.ws = Buffer(torch.zeros(max(16, self.ws_bytes), dtype=torch.uint8, device="cuda"))
        self.position = Buffer(torch.tensor([c["length"] - 1], dtype=torch.int32, device="cuda"))


class Step:
    """Launches captured in a graph, replayed per pass."""

    def __init__(self, fn):
        torch.cuda.synchronize()
        self.graph = dev.Graph.capture(fn)

    def __call__(self):
        self.graph.launch()

    def __del__(self):
        try:
            self.graph.close()
        except Exception:
            pass


def _supported(call, *args):
    """Runs a fused launch; False where the engine has none for the shape."""
    try:
        call(*args)
        return True
    except hip.CitlaliError as e:
        if e.status != hip._lib.ERR_UNSUPPORTED:
            raise
        return False


def _enqueue_layer(c, lay, s, x, x_alt, pending):
    """One layer's launches, as forward_token makes them: the fused launch
    where there is one, the separate ones elsewhere.  `pending` is the
    previous layer's FFN output, not yet added to the residual `x`; returns
    the residual buffers in their new order (the layer's FFN output is left
    in s.ffn_out)."""
    h, f, nh, nkv, hd = c["hidden"], c["ffn"], c["heads"], c["kv_heads"], c["head_dim"]
    t, w, rows = lay.types, lay.w, {n: lay.shapes[n][0] for n in lay.shapes}
    qkv, outs = ("q", "k", "v"), (s.q, s.k, s.v)
    if _supported(dev.matvec_group_norm, [t[n] for n in qkv], [w[n] for n in qkv], x, pending, lay.attn_norm,
                  x_alt if pending else None, EPS, outs, [rows[n] for n in qkv], h):
        if pending:
            x, x_alt = x_alt, x
    else:
        if pending:
            dev.add_rms_norm(x, pending, lay.attn_norm, s.norm, h, EPS)
        else:
            dev.rms_norm(x, lay.attn_norm, s.norm, h, EPS)
        if not _supported(dev.matvec_group, [t[n] for n in qkv], [w[n] for n in qkv], s.norm, outs,
                          [rows[n] for n in qkv], h):
            for n, y in zip(qkv, outs):
                dev.matvec(t[n], w[n], s.norm, y, h, rows[n])
    for n, y in zip(qkv, outs):
        if n in lay.bias:
            dev.add_bias_inplace(y, lay.bias[n], rows[n])
    plan = dev.attention_plan_length(c["length"], c["max_context"])
    if not _supported(dev.qk_norm_rope_store_attention, s.q, s.k, s.v, lay.q_norm, lay.k_norm, nh, nkv, hd,
                      s.position, plan, c["max_context"], THETA, EPS, lay.k_cache, lay.v_cache, s.ws, s.ws_bytes,
                      s.attn):
        dev.qk_norm_rope_store_at(s.q, s.k, s.v, lay.q_norm, lay.k_norm, nh, nkv, hd, s.position, c["max_context"],
                                  THETA, EPS, lay.k_cache, lay.v_cache)
        dev.attention_batched(s.q, lay.k_cache, lay.v_cache, 0, s.position, plan, 1, nh, nkv, hd, s.ws, s.ws_bytes,
                              s.attn)
    dev.matvec(t["o"], w["o"], s.attn, s.proj, nh * hd, h)
    if _supported(dev.matvec_gate_up_swiglu_norm, t["gate"], w["gate"], w["up"], x, s.proj, lay.ffn_norm, x_alt, EPS,
                  s.act, h, f):
        x, x_alt = x_alt, x
    else:
        dev.add_rms_norm(x, s.proj, lay.ffn_norm, s.norm, h, EPS)
        if not _supported(dev.matvec_gate_up_swiglu, t["gate"], w["gate"], w["up"], s.norm, s.act, h, f):
            dev.matvec(t["gate"], w["gate"], s.norm, s.gate, h, f)
            dev.matvec(t["up"], w["up"], s.norm, s.up, h, f)
            dev.swiglu(s.gate, s.up, s.act, f)
    dev.matvec(t["down"], w["down"], s.act, s.ffn_out, f, h)
    return x, x_alt


# ---------------------------------------------------------------- prepare / run
def prepare(case, seed):
    _library()
    c, g = dict(case), _gen(seed)
    kind = c["kind"]
    st = {"case": c}
    if kind == "matvec":
        st["w"] = Buffer(_weight(g, c["quant"], c["rows"], c["cols"]))
        st["x"] = Buffer(_hidden_state(g, c["cols"]))
        st["y"] = Buffer(torch.zeros(c["rows"], dtype=torch.float32 if c["f32"] else torch.float16, device="cuda"))
    elif kind == "head":
        st["w"] = Buffer(_weight(g, c["quant"], c["rows"], c["cols"], 3.0))
        st["x"], st["delta"] = Buffer(_hidden_state(g, c["cols"])), Buffer(_normal(g, c["cols"]))
        st["norm"], st["sum"] = Buffer(_norm_weight(g, c["cols"])), _half(c["cols"])
        st["y"] = Buffer(torch.zeros(c["rows"], dtype=torch.float32, device="cuda"))
    elif kind == "attention":
        st["q"] = Buffer(_normal(g, c["heads"], c["head_dim"]))
        st["k"], st["v"] = (Buffer(_normal(g, c["max_context"], c["kv_heads"], c["head_dim"])) for _ in range(2))
        st["scores"] = Buffer(torch.zeros(c["heads"] * c["max_context"], dtype=torch.float32, device="cuda"))
        st["y"] = _half(c["heads"], c["head_dim"])
    elif kind == "batch":
        rows = (c["nseq"], c["longest"], c["kv_heads"], c["head_dim"])
        st["q"] = Buffer(_normal(g, c["nseq"], c["heads"], c["head_dim"]))
        st["k"], st["v"] = Buffer(_normal(g, *rows)), Buffer(_normal(g, *rows))
        st["positions"] = Buffer(torch.tensor([n - 1 for n in _lengths(c, seed)], dtype=torch.int32, device="cuda"))
        st["ws_bytes"] = dev.attention_workspace_bytes(c["longest"], c["nseq"], c["heads"], c["kv_heads"],
                                                       c["head_dim"])
        st["ws"] = Buffer(torch.zeros(max(16, st["ws_bytes"]), dtype=torch.uint8, device="cuda"))
        st["y"] = _half(c["nseq"], c["heads"], c["head_dim"])
    elif kind == "load":
        for q in ("q4k", "q6k"):
            n = (c[q] + 255) // 256
            st[q] = Buffer(_weight(g, q, n, 256, 16.0 / math.sqrt(4096)))
            st["y_" + q] = _half(c[q])
    elif kind == "layer":
        s, lay = Scratch(c), Layer(g, c)
        s.x.tensor.copy_(_hidden_state(g, c["hidden"]))
        st.update(s=s, layer=lay)
        st["h"] = []
        st["step"] = Step(lambda: st["h"].append(_enqueue_layer(c, lay, s, s.x, s.x_alt, None)))
    else:
        s, layers = Scratch(c), [Layer(g, c) for _ in range(c["layers"])]
        st.update(s=s, layers=layers)
        st["embedding"] = Buffer(_weight(g, "q6k", c["vocab"], c["hidden"], math.sqrt(c["hidden"])))
        st["output"] = Buffer(_weight(g, "q6k", c["vocab"], c["hidden"], 3.0))
        st["norm"] = Buffer(_norm_weight(g, c["hidden"]))
        st["token"] = Buffer(torch.randint(0, c["vocab"], (1,), generator=g, device="cuda", dtype=torch.int32))
        st["logits"] = Buffer(torch.zeros(c["vocab"], dtype=torch.float32, device="cuda"))
        st["next"] = Buffer(torch.zeros(1, dtype=torch.int32, device="cuda"))

        def step():
            dev.embed_q6k_at(st["embedding"], st["token"], c["vocab"], s.x, c["hidden"])
            x, x_alt = s.x, s.x_alt
            for i, lay in enumerate(layers):
                x, x_alt = _enqueue_layer(c, lay, s, x, x_alt, s.ffn_out if i else None)
            if not _supported(dev.matvec_norm, "q6k", st["output"], x, s.ffn_out, st["norm"], x_alt, EPS,
                              st["logits"], c["hidden"], c["vocab"], True):
                dev.add_rms_norm(x, s.ffn_out, st["norm"], s.norm, c["hidden"], EPS)
                dev.matvec("q6k", st["output"], s.norm, st["logits"], c["hidden"], c["vocab"], f32_out=True)
            dev.argmax(st["logits"], c["vocab"], st["next"])

        st["step"] = Step(step)
    return st


def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "matvec":
        dev.matvec(c["quant"], st["w"], st["x"], st["y"], c["cols"], c["rows"], f32_out=c["f32"])
        return st["y"].tensor
    if kind == "head":
        dev.matvec_norm(c["quant"], st["w"], st["x"], st["delta"], st["norm"], st["sum"], EPS, st["y"], c["cols"],
                        c["rows"], f32_out=True)
        return st["y"].tensor, st["sum"].tensor
    if kind == "attention":
        dev.attention(st["q"], st["k"], st["v"], st["scores"], st["y"], c["length"] - 1, c["max_context"], c["heads"],
                      c["kv_heads"], c["head_dim"])
        return st["y"].tensor
    if kind == "batch":
        dev.attention_batched(st["q"], st["k"], st["v"], c["longest"] * c["kv_heads"] * c["head_dim"],
                              st["positions"], c["longest"], c["nseq"], c["heads"], c["kv_heads"], c["head_dim"],
                              st["ws"], st["ws_bytes"], st["y"])
        return st["y"].tensor
    if kind == "load":
        dev.dequant_f16("q4k", st["q4k"], c["q4k"], st["y_q4k"])
        dev.dequant_f16("q6k", st["q6k"], c["q6k"], st["y_q6k"])
        return st["y_q4k"].tensor, st["y_q6k"].tensor
    st["step"]()
    p = c["length"] - 1
    if kind == "layer":
        s, lay = st["s"], st["layer"]
        return {"residual": st["h"][0][0].tensor, "ffn": s.ffn_out.tensor, "attn": s.attn.tensor,
                "k": lay.k_cache.tensor[p], "v": lay.v_cache.tensor[p]}
    # the pick is a function of the logits, which are what can be compared
    return {"logits": st["logits"].tensor, "k": st["layers"][-1].k_cache.tensor[p],
            "v": st["layers"][-1].v_cache.tensor[p]}


def _lengths(c, seed):
    g = torch.Generator().manual_seed(int(seed) * 31 + 5)
    n = torch.randint(c["shortest"], c["longest"] + 1, (c["nseq"],), generator=g).tolist()
    n[0] = c["longest"]
    return n


# ---------------------------------------------------------------- work
def _matrix_bytes(quant, rows, cols):
    return rows * cols // 256 * BLOCK_BYTES[quant]


def _layer_work(c):
    nq, nkv, h, f = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"], c["hidden"], c["ffn"]
    t = MIXES[c["mix"]]
    shapes = dict(q=(nq, h), k=(nkv, h), v=(nkv, h), o=(h, nq), gate=(f, h), up=(f, h), down=(h, f))
    b = sum(_matrix_bytes(t[n], *shapes[n]) for n in shapes)
    fl = sum(2 * r * k for r, k in shapes.values())
    b += 2 * c["length"] * nkv * 2 + 6 * h
    fl += 4 * c["length"] * nq
    return b, fl


def work(case):
    c = case
    kind = c["kind"]
    if kind in ("matvec", "head"):
        out = 4 if kind == "head" or c["f32"] else 2
        return {"bytes": _matrix_bytes(c["quant"], c["rows"], c["cols"]) + 2 * c["cols"] + out * c["rows"],
                "flops": 2 * c["rows"] * c["cols"]}
    if kind == "attention":
        return {"bytes": 4 * c["length"] * c["kv_heads"] * c["head_dim"] + 4 * c["heads"] * c["head_dim"],
                "flops": 4 * c["length"] * c["heads"] * c["head_dim"]}
    if kind == "batch":
        n = c["nseq"] * (c["shortest"] + c["longest"]) / 2   # mean total length
        return {"bytes": 4 * n * c["kv_heads"] * c["head_dim"] + 4 * c["nseq"] * c["heads"] * c["head_dim"],
                "flops": 4 * n * c["heads"] * c["head_dim"]}
    if kind == "load":
        n = c["q4k"] + c["q6k"]
        return {"bytes": c["q4k"] * 144 / 256 + c["q6k"] * 210 / 256 + 2 * n, "flops": 3 * n}
    b, fl = _layer_work(c)
    if kind == "model":
        b, fl = b * c["layers"], fl * c["layers"]
        b += _matrix_bytes("q6k", c["vocab"], c["hidden"]) + 4 * c["vocab"]
        fl += 2 * c["vocab"] * c["hidden"]
    return {"bytes": b, "flops": fl}


def tolerance(case):
    kind = case["kind"]
    if kind == "load":
        return "exact"                       # the host loader's rounding, bit for bit
    # about four times what two correct implementations were seen to differ by
    # (each measured against 64 bits: fp32 sums 2e-6, one fp16 rounding 2e-4,
    # a layer's store points 6e-4, 28 layers 2e-3)
    if kind == "matvec" and case["f32"]:
        return {"rel": 1e-5, "max": 1e-3}    # fp32 sums
    if kind == "head":
        return {"rel": 1.3e-3, "max": 3e-2}  # fp16 normed input, fp32 sums
    if kind == "layer":
        return {"rel": 2.5e-3, "max": 6e-2}  # six fp16 store points in a row
    if kind == "model":
        return {"rel": 1.2e-2, "max": 3e-1}  # fp16 store points through every layer
    return {"rel": 1e-3, "max": 2e-2}        # fp32 sums, one fp16 rounding


# ---------------------------------------------------------------- 64-bit results
def _f64_blocks(quant, b):
    """Values of K-quant blocks, [n][256] float64."""
    n = b.shape[0]
    b32 = b.to(torch.int32)
    if quant == "q4k":
        d = b[:, 0:2].contiguous().view(torch.float16).double()
        dmin = b[:, 2:4].contiguous().view(torch.float16).double()
        s = b32[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        m = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b32[:, 16:].view(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(n, 8, 32).double()
        return ((d * sc).unsqueeze(2) * q - (dmin * m).unsqueeze(2)).view(n, 256)
    ql, qh = b32[:, 0:128].view(n, 2, 2, 32), b32[:, 128:192].view(n, 2, 1, 32)
    lo = torch.cat([ql & 15, ql >> 4], 2)                                      # [n][half][part][32]
    hi = torch.cat([(qh >> (2 * p)) & 3 for p in range(4)], 2)
    sc = b[:, 192:208].contiguous().view(torch.int8).double().view(n, 2, 4, 2, 1)
    d = b[:, 208:210].contiguous().view(torch.float16).double().view(n, 1, 1, 1, 1)
    return (d * sc * ((lo | (hi << 4)) - 32).double().view(n, 2, 4, 2, 16)).view(n, 256)


def _f64_matvec(quant, w, x):
    """Rows of `w` times x (float64)."""
    cols = x.numel()
    if quant == "fp16":
        return torch.cat([p.double() @ x for p in w.split(max(1, (1 << 26) // cols))])
    nb = cols // 256
    w = w.view(-1, nb, w.shape[-1])
    step = max(1, (1 << 25) // cols)
    return torch.cat([_f64_blocks(quant, p.reshape(-1, p.shape[-1])).view(-1, cols) @ x for p in w.split(step)])


def _f64_norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _f64_rope(x, position):
    half = x.shape[-1] // 2
    i = torch.arange(half, device=x.device, dtype=torch.float64)
    a = position * THETA ** (-2 * i / x.shape[-1])
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat([lo * a.cos() - hi * a.sin(), lo * a.sin() + hi * a.cos()], -1)


def _f64_attention(q, k, v):
    """q [heads][hd], k / v [L][kv][hd] -> [heads][hd]."""
    kv = k.shape[1]
    group = q.shape[0] // kv
    out = []
    for j in range(kv):
        s = q[j * group:(j + 1) * group].double() @ k[:, j].double().t().contiguous() / math.sqrt(q.shape[1])
        out.append(torch.softmax(s, -1) @ v[:, j].double())
    return torch.cat(out)


def _f64_layer(c, lay, x):
    """(residual after attention, ffn output, attention output, k row, v row)"""
    p, hd = c["length"] - 1, c["head_dim"]
    n = _f64_norm(x, lay.attn_norm.tensor)
    q, k, v = (_f64_matvec(lay.types[m], lay.w[m].tensor, n) for m in ("q", "k", "v"))
    if lay.bias:
        q, k, v = (y + lay.bias[m].tensor.double() for y, m in ((q, "q"), (k, "k"), (v, "v")))
    q, k, v = (y.view(-1, hd) for y in (q, k, v))
    if lay.q_norm is not None:
        q, k = _f64_norm(q, lay.q_norm.tensor), _f64_norm(k, lay.k_norm.tensor)
    q, k = _f64_rope(q, p), _f64_rope(k, p)
    kc = torch.cat([lay.k_cache.tensor[:p].double(), k[None]])
    vc = torch.cat([lay.v_cache.tensor[:p].double(), v[None]])
    attn = _f64_attention(q, kc, vc).reshape(-1)
    h = x + _f64_matvec(lay.types["o"], lay.w["o"].tensor, attn)
    n = _f64_norm(h, lay.ffn_norm.tensor)
    g, u = (_f64_matvec(lay.types[m], lay.w[m].tensor, n) for m in ("gate", "up"))
    return h, _f64_matvec(lay.types["down"], lay.w["down"].tensor, g * torch.sigmoid(g) * u), attn, k, v


def exact(case, seed):
    st = prepare(case, seed)
    torch.cuda.synchronize()
    c = st["case"]
    kind = c["kind"]
    if kind == "matvec":
        return _f64_matvec(c["quant"], st["w"].tensor, st["x"].tensor.double())
    if kind == "head":
        s = st["x"].tensor.double() + st["delta"].tensor.double()
        return _f64_matvec(c["quant"], st["w"].tensor, _f64_norm(s, st["norm"].tensor)), s
    if kind == "attention":
        n = c["length"]
        return _f64_attention(st["q"].tensor, st["k"].tensor[:n], st["v"].tensor[:n])
    if kind == "batch":
        return torch.stack([_f64_attention(st["q"].tensor[i], st["k"].tensor[i, :n], st["v"].tensor[i, :n])
                            for i, n in enumerate(_lengths(c, seed))])
    if kind == "load":
        return tuple(torch.cat([_f64_blocks(q, p).view(-1) for p in st[q].tensor.split(1 << 17)])[:c[q]]
                     for q in ("q4k", "q6k"))
    if kind == "layer":
        h, ffn, attn, k, v = _f64_layer(c, st["layer"], st["s"].x.tensor.double())
        return {"residual": h, "ffn": ffn, "attn": attn, "k": k, "v": v}
    nb = c["hidden"] // 256
    t = int(st["token"].tensor[0])
    x = _f64_blocks("q6k", st["embedding"].tensor[t * nb:(t + 1) * nb]).view(-1)
    for lay in st["layers"]:
        h, ffn, _, k, v = _f64_layer(c, lay, x)
        x = h + ffn
    return {"logits": _f64_matvec("q6k", st["output"].tensor, _f64_norm(x, st["norm"].tensor)), "k": k, "v": v}
