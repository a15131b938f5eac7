"""Cases of the backend's work at the sizes its users run: prefill and decode of Phi-2 / Phi-3-mini sized models in f16 and
bf16, a Whisper-tiny encoder in f32, long and ragged prompts, batches, and the GroupNorm of a convolutional front end.

listed() names the cases, draw() gives more of the same ranges, prepare() makes what a program has in hand before the calls
(device buffers filled from the seed, output buffers, graph inputs) and run() is one pass through the public entry points
(ratchet_amd.Device for the kernels, ratchet_amd.host for the lazy Tensor graphs).  A pass enqueues on the device's stream
and returns; only the graph case waits, where it downloads its results as its users do."""
import numpy as np
import torch

from ratchet_amd import Device, _lib, host

DT = {"f32": _lib.F32, "f16": _lib.F16, "bf16": _lib.BF16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i32": torch.int32}
#: attention and MLP geometry of one layer: heads, head dim, rotary width, hidden width, MLP width
LAYER = {"phi2": (32, 80, 32, 2560, 10240), "phi3": (32, 96, 96, 3072, 8192)}
EPS = 1e-5
LARGEST = 2.2e9          # bytes of the largest listed case

_open = {}


def _device():
    if "dev" not in _open:
        _open["dev"] = Device(0)
    return _open["dev"]


def _graph_device():
    if "graph" not in _open:
        _open["graph"] = host.HostDevice(0)
    return _open["graph"]


class _Window:
    """What torch needs to see a device buffer of the library without a copy."""

    def __init__(self, buf, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": buf.shape, "typestr": typestr, "data": (buf.ptr.value, False), "version": 2}


def _seen(buf):
    code = buf.dt
    t = torch.as_tensor(_Window(buf, {_lib.F32: "<f4", _lib.F16: "<f2", _lib.BF16: "<i2", _lib.I32: "<i4"}[code]), device="cuda")
    return t.view(torch.bfloat16) if code == _lib.BF16 else t


class _Maker:
    """Buffers of one state: inputs drawn from the seed, outputs left as they are."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(int(seed))
        self.dev = _device()

    def normal(self, shape, dtype, std=1.0, mean=0.0):
        buf = self.dev.empty(shape, DT[dtype])
        view, flat = _seen(buf).view(-1), 1 << 26
        for at in range(0, view.numel(), flat):                # in pieces: the f32 draws of a large tensor need not all exist at once
            part = view[at:at + flat]
            part.copy_(torch.randn(part.numel(), generator=self.gen, device="cuda").mul_(std).add_(mean))
        return buf

    def causal(self, queries, keys, dtype):
        """-inf above the diagonal of the last `queries` rows of a causal mask over `keys`"""
        buf = self.dev.empty((queries, keys), DT[dtype])
        q = torch.arange(queries, device="cuda").view(-1, 1) + (keys - queries)
        k = torch.arange(keys, device="cuda").view(1, -1)
        _seen(buf).copy_(torch.where(k > q, float("-inf"), 0.0))
        return buf

    def ints(self, n, below):
        buf = self.dev.empty((n,), _lib.I32)
        _seen(buf).copy_(torch.randint(0, below, (n,), generator=self.gen, device="cuda", dtype=torch.int32))
        return buf

    def empty(self, shape, dtype):
        buf = self.dev.empty(shape, DT[dtype])
        _seen(buf).zero_()
        return buf


# ---------------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # one token through a Phi-2 layer with 2047 tokens in the KV cache: nine small launches, the latency of a generated token
        {"name": "decode_phi2_f16", "kind": "decode", "layer": "phi2", "dtype": "f16", "context": 2047},
        # the same ops as lazy graphs built, planned, resolved and downloaded for each token, as the models do
        {"name": "graph_phi2_f16", "kind": "graph", "layer": "phi2", "tokens": 1, "context": 2047},
        # MLP of a Whisper-tiny encoder layer over eight 30 s windows: bias, GELU, LayerNorm, all f32
        {"name": "encoder_mlp_f32", "kind": "encoder_mlp", "batch": 8, "frames": 1500, "width": 384},
        # attention of the same encoder, one window: heads apart and together again, softmax of [1,6,1500,1500]
        {"name": "encoder_attention_f32", "kind": "encoder_attention", "batch": 1, "frames": 1500, "heads": 6},
        # LayerNorm of a 2048-token Phi-2 prompt in the reference's f16 arithmetic
        {"name": "layer_norm_2048x2560_f16", "kind": "norm", "norm": "layer", "dtype": "f16", "rows": 2048, "cols": 2560},
        # RMSNorm of four 4096-token Phi-3 prompts in bf16
        {"name": "rms_norm_16384x3072_bf16", "kind": "norm", "norm": "rms", "dtype": "bf16", "rows": 16384, "cols": 3072},
        # a Phi-3 layer over a 2048-token prompt the way the models emit it (full -> op -> cast in one launch each)
        {"name": "prefill_phi3_2048_bf16", "kind": "prefill", "layer": "phi3", "dtype": "bf16", "tokens": 2048},
        # causal attention weights of a 4096-token Phi-3 prompt, mask and softmax in f16: the largest tensor here
        {"name": "scores_4096_f16", "kind": "scores", "dtype": "f16", "heads": 32, "queries": 4096, "keys": 4096, "mask": True},
        # the same of a prompt of 1001 tokens: no row starts on a vector boundary
        {"name": "scores_1001_f16", "kind": "scores", "dtype": "f16", "heads": 32, "queries": 1001, "keys": 1001, "mask": True},
        # the last 2048 tokens of an 8192-token prompt over all its keys
        {"name": "scores_2048x8192_f16", "kind": "scores", "dtype": "f16", "heads": 8, "queries": 2048, "keys": 8192, "mask": True},
        # keys of four 2048-token Phi-2 prompts: heads apart, rotary, into the KV cache, transposed for the scores
        {"name": "keys_4x2048x80_f16", "kind": "keys", "dtype": "f16", "batch": 4, "heads": 32, "tokens": 2048, "past": 0, "dim": 80, "rotary": 32},
        # GroupNorm behind the convolutions of sixteen 30 s windows
        {"name": "group_norm_16x512x3000_f16", "kind": "group_norm", "dtype": "f16", "batch": 16, "channels": 512, "length": 3000, "groups": 32},
    ]


def _spread(rng, low, high, step=1):
    """log-uniform over [low, high], half of the time a multiple of `step`"""
    v = int(round(low * (high / low) ** rng.random()))
    if step > 1 and rng.random() < 0.5:
        v = max(low, v // step * step)
    return max(low, min(high, v))


def draw(rng):
    while True:
        kind = rng.choice(["decode", "graph", "encoder_mlp", "encoder_attention", "norm", "norm", "prefill", "scores", "scores", "keys", "group_norm"])
        half = rng.choice(["f16", "bf16"])
        layer = rng.choice(sorted(LAYER))
        if kind == "decode":
            c = {"layer": layer, "dtype": half, "context": _spread(rng, 64, 8000)}
        elif kind == "graph":
            c = {"layer": layer, "tokens": _spread(rng, 1, 32), "context": _spread(rng, 64, 4000)}
        elif kind == "encoder_mlp":
            c = {"batch": _spread(rng, 1, 16), "frames": rng.choice([1500, rng.randint(100, 1500)]), "width": rng.choice([384, 512, 768])}
        elif kind == "encoder_attention":
            c = {"batch": rng.randint(1, 4), "frames": rng.choice([1500, rng.randint(100, 1500)]), "heads": rng.choice([6, 8, 12])}
        elif kind == "norm":
            c = {"norm": rng.choice(["layer", "rms"]), "dtype": half, "rows": _spread(rng, 256, 32768, 64), "cols": _spread(rng, 384, 5120, 128)}
        elif kind == "prefill":
            c = {"layer": "phi3", "dtype": half, "tokens": _spread(rng, 64, 3500, 64)}
        elif kind == "scores":
            queries = _spread(rng, 16, 4096, 16)
            c = {"dtype": half, "heads": rng.choice([8, 16, 32]), "queries": queries, "keys": queries if rng.random() < 0.6 else _spread(rng, queries, 8192, 16),
                 "mask": rng.random() < 0.75}
        elif kind == "keys":
            dim, rotary = rng.choice([(64, 64), (80, 32), (96, 96), (128, 128)])
            c = {"dtype": rng.choice(["f16", "bf16", "f32"]), "batch": rng.randint(1, 4), "heads": rng.choice([8, 32]), "tokens": _spread(rng, 32, 4096, 32),
                 "past": rng.choice([0, rng.randint(1, 2048)]), "dim": dim, "rotary": rotary}
        else:
            c = {"dtype": rng.choice(["f16", "f32"]), "batch": _spread(rng, 1, 16), "channels": rng.choice([256, 320, 512, 640]), "length": _spread(rng, 64, 16384, 64),
                 "groups": 32}
        c["kind"] = kind
        cost = work(c)["bytes"] * (2.5 if kind == "encoder_mlp" or c.get("keys", 0) > 4096 else 1.5)      # bytes of these take longer than a copy's
        if cost < LARGEST:
            return c


# ------------------------------------------------------------------------------------------------------------- prepare
def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_decode(c, seed):
    heads, dim, rotary, hidden, wide = LAYER[c["layer"]]
    m, t, d = _Maker(seed), c["context"], c["dtype"]
    s = {"run": _run_decode, "rotary": rotary, "at": t,
         "table": m.normal((4096, hidden), d), "ids": m.ints(1, 4096), "w": m.normal((hidden,), "f32", 0.02, 1.0), "b": m.normal((hidden,), "f32", 0.02),
         "q": m.normal((1, heads, 1, dim), d), "k": m.normal((1, heads, 1, dim), d), "v": m.normal((1, heads, 1, dim), d),
         "kc": m.normal((1, heads, t + 1, dim), d), "vc": m.normal((1, heads, t + 1, dim), d),
         "scores": m.normal((1, heads, 1, t + 1), d, 2.0), "ff": m.normal((1, wide), d)}
    out = {"x": (1, hidden), "h": (1, hidden), "q": (1, heads, 1, dim), "k": (1, heads, 1, dim), "keys": (1, heads, t + 1, dim),
           "values": (1, heads, t + 1, dim), "probs": (1, heads, 1, t + 1), "act": (1, wide), "res": (1, hidden)}
    s["out"] = {k: m.empty(v, d) for k, v in out.items()}
    s["seen"] = {k: _seen(v) for k, v in list(s["out"].items()) + [("kc", s["kc"]), ("vc", s["vc"])]}
    return s


def _run_decode(s):
    dev, o = _device(), s["out"]
    dev.index_select(s["table"], s["ids"], 0, out=o["x"])
    dev.norm_via_f32("layer", o["x"], s["w"], s["b"], EPS, out=o["h"])
    dev.rope(s["q"], s["rotary"], 10000.0, s["at"], out=o["q"])
    dev.rope(s["k"], s["rotary"], 10000.0, s["at"], out=o["k"])
    dev.cache(s["kc"], o["k"], 2, s["at"], out=o["keys"])
    dev.cache(s["vc"], s["v"], 2, s["at"], out=o["values"])
    dev.softmax_via_f32(s["scores"], None, out=o["probs"])
    dev.unary_via_f32("gelu", s["ff"], out=o["act"])
    dev.binary("add", o["x"], o["h"], out=o["res"])
    return s["seen"]


def _prepare_graph(c, seed):
    heads, dim, rotary, hidden, wide = LAYER[c["layer"]]
    gen, n, t, dev = torch.Generator(device="cuda"), c["tokens"], c["context"], _graph_device()
    gen.manual_seed(int(seed))

    def up(shape, std=1.0, mean=0.0, kind=torch.float16):
        return host.Tensor.from_numpy(torch.randn(shape, generator=gen, device="cuda").mul_(std).add_(mean).to(kind).cpu().numpy(), dev)

    ids = torch.randint(0, 4096, (n,), generator=gen, device="cuda", dtype=torch.int32).cpu().numpy()
    return {"run": _run_graph, "rotary": rotary, "at": t, "table": up((4096, hidden)), "ids": host.Tensor.from_numpy(ids, dev),
            "w": up((hidden,), 0.02, 1.0, torch.float32), "b": up((hidden,), 0.02, 0.0, torch.float32), "k": up((1, heads, n, dim)),
            "scores": up((1, heads, n, t + n), 2.0), "ff": up((n, wide))}


def _run_graph(s):
    x = s["table"].index_select(s["ids"], 0)
    h = x.full().layer_norm(s["w"], s["b"], EPS).cast(_lib.F16)
    roots = [x.add(h), s["k"].full().rope(s["rotary"], 10000.0, s["at"]).cast(_lib.F16), s["scores"].full().softmax(3).cast(_lib.F16),
             s["ff"].full().gelu().cast(_lib.F16)]
    return [r.resolve().to_numpy() for r in roots]


def _prepare_encoder_mlp(c, seed):
    m, b, t, n = _Maker(seed), c["batch"], c["frames"], c["width"]
    s = {"run": _run_encoder_mlp, "ff": m.normal((b, t, 4 * n), "f32"), "ffb": m.normal((4 * n,), "f32", 0.02), "x": m.normal((b, t, n), "f32"),
         "w": m.normal((n,), "f32", 0.02, 1.0), "b": m.normal((n,), "f32", 0.02)}
    s["out"] = {"biased": m.empty((b, t, 4 * n), "f32"), "act": m.empty((b, t, 4 * n), "f32"), "normed": m.empty((b, t, n), "f32")}
    s["seen"] = {k: _seen(v) for k, v in s["out"].items()}
    return s


def _run_encoder_mlp(s):
    dev, o = _device(), s["out"]
    dev.binary("add", s["ff"], s["ffb"], out=o["biased"])
    dev.unary("gelu", o["biased"], out=o["act"])
    dev.layer_norm(s["x"], s["w"], s["b"], EPS, out=o["normed"])
    return s["seen"]


def _prepare_encoder_attention(c, seed):
    m, b, t, h = _Maker(seed), c["batch"], c["frames"], c["heads"]
    s = {"run": _run_encoder_attention, "q": m.normal((b, t, h, 64), "f32"), "scores": m.normal((b, h, t, t), "f32", 3.0), "mixed": m.normal((b, h, t, 64), "f32")}
    s["out"] = {"apart": m.empty((b, h, t, 64), "f32"), "probs": m.empty((b, h, t, t), "f32"), "together": m.empty((b, t, h, 64), "f32")}
    s["seen"] = {k: _seen(v) for k, v in s["out"].items()}
    return s


def _run_encoder_attention(s):
    dev, o = _device(), s["out"]
    dev.permute(s["q"], (0, 2, 1, 3), out=o["apart"])
    dev.softmax(s["scores"], out=o["probs"])
    dev.permute(s["mixed"], (0, 2, 1, 3), out=o["together"])
    return s["seen"]


def _prepare_norm(c, seed):
    m, shape, d = _Maker(seed), (c["rows"], c["cols"]), c["dtype"]
    s = {"run": _run_norm, "norm": c["norm"], "x": m.normal(shape, d), "w": m.normal((c["cols"],), d, 0.02, 1.0), "b": m.normal((c["cols"],), d, 0.02)}
    s["y"] = m.empty(shape, d)
    s["seen"] = _seen(s["y"])
    return s


def _run_norm(s):
    dev = _device()
    if s["norm"] == "layer":
        dev.layer_norm(s["x"], s["w"], s["b"], EPS, out=s["y"])
    else:
        dev.rms_norm(s["x"], s["w"], EPS, out=s["y"])
    return s["seen"]


def _prepare_prefill(c, seed):
    heads, dim, rotary, hidden, wide = LAYER[c["layer"]]
    m, t, d = _Maker(seed), c["tokens"], c["dtype"]
    s = {"run": _run_prefill, "rotary": rotary, "x": m.normal((1, t, hidden), d), "w": m.normal((hidden,), "f32", 0.02, 1.0),
         "q": m.normal((1, heads, t, dim), d), "scores": m.normal((1, heads, t, t), d, 2.0), "mask": m.causal(t, t, d),
         "gate_up": m.normal((t, 2 * wide), d), "attn": m.normal((1, t, hidden), d, 0.5), "wide": wide, "tokens": t}
    s["out"] = {"normed": m.empty((1, t, hidden), d), "q": m.empty((1, heads, t, dim), d), "probs": m.empty((1, heads, t, t), d),
                "gated": m.empty((t, wide), d), "res": m.empty((1, t, hidden), d)}
    s["gate"], s["up"] = s["gate_up"].reshape((t, 2 * wide)), s["gate_up"].view(wide, ((2 * t - 1) * wide,))
    s["seen"] = {k: _seen(v) for k, v in s["out"].items()}
    return s


def _run_prefill(s):
    dev, o = _device(), s["out"]
    dev.norm_via_f32("rms", s["x"], s["w"], None, EPS, out=o["normed"])
    dev.rope(s["q"], s["rotary"], 10000.0, 0, out=o["q"])
    dev.softmax_via_f32(s["scores"], s["mask"], out=o["probs"])
    dev.gated_mul_via_f32("silu", s["gate"], s["up"], s["tokens"], s["wide"], 2 * s["wide"], 2 * s["wide"], out=o["gated"])
    dev.binary("add", s["x"], s["attn"], out=o["res"])
    return s["seen"]


def _prepare_scores(c, seed):
    # N(0, 1) for long rows: the reference arithmetic subtracts no maximum, and the f16 sum of 8192 exp(N(0, 2)) would overflow
    m, shape, d = _Maker(seed), (1, c["heads"], c["queries"], c["keys"]), c["dtype"]
    s = {"run": _run_scores, "x": m.normal(shape, d, 2.0 if c["keys"] <= 4096 else 1.0), "mask": m.causal(c["queries"], c["keys"], d) if c["mask"] else None, "y": m.empty(shape, d)}
    s["seen"] = _seen(s["y"])
    return s


def _run_scores(s):
    if s["mask"] is None:
        _device().softmax(s["x"], out=s["y"])
    else:
        _device().softmax_masked(s["x"], s["mask"], out=s["y"])
    return s["seen"]


def _prepare_keys(c, seed):
    m, b, h, t, p, n, d = _Maker(seed), c["batch"], c["heads"], c["tokens"], c["past"], c["dim"], c["dtype"]
    s = {"run": _run_keys, "rotary": c["rotary"], "past": p, "x": m.normal((b, t, h, n), d), "cache": m.normal((b, h, p + t, n), d)}
    s["out"] = {"apart": m.empty((b, h, t, n), d), "turned": m.empty((b, h, t, n), d), "keys": m.empty((b, h, p + t, n), d), "across": m.empty((b, h, n, p + t), d)}
    s["seen"] = {k: _seen(v) for k, v in list(s["out"].items()) + [("cache", s["cache"])]}
    return s


def _run_keys(s):
    dev, o = _device(), s["out"]
    dev.permute(s["x"], (0, 2, 1, 3), out=o["apart"])
    dev.rope(o["apart"], s["rotary"], 10000.0, s["past"], out=o["turned"])
    dev.cache(s["cache"], o["turned"], 2, s["past"], out=o["keys"])
    dev.permute(o["keys"], (0, 1, 3, 2), out=o["across"])
    return s["seen"]


def _prepare_group_norm(c, seed):
    m, shape, d = _Maker(seed), (c["batch"], c["channels"], c["length"]), c["dtype"]
    s = {"run": _run_group_norm, "groups": c["groups"], "x": m.normal(shape, d), "w": m.normal((c["channels"],), d, 0.02, 1.0),
         "b": m.normal((c["channels"],), d, 0.02), "y": m.empty(shape, d)}
    s["seen"] = _seen(s["y"])
    return s


def _run_group_norm(s):
    _device().group_norm(s["x"], s["groups"], s["w"], s["b"], EPS, out=s["y"])
    return s["seen"]


# ---------------------------------------------------------------------------------------------------- work, tolerance
def work(case):
    """each call's operands read once and its results written once"""
    c, kind = case, case["kind"]
    e = BYTES[c.get("dtype", "f32")]
    if kind in ("decode", "graph", "prefill"):
        heads, dim, _, hidden, wide = LAYER[c["layer"]]
    if kind == "decode":
        n = 2 * hidden + 2 * hidden + 4 * heads * dim + 2 * heads * dim * (2 * c["context"] + 3) + 2 * heads * (c["context"] + 1) + 2 * wide + 3 * hidden
        return {"bytes": n * e + 8 * hidden, "flops": 10.0 * (hidden + heads * c["context"] + wide)}
    if kind == "graph":
        t = c["tokens"]
        n = 2 * t * hidden + 2 * t * hidden + 3 * t * hidden + 2 * heads * t * dim + 2 * heads * t * (c["context"] + t) + 2 * t * wide
        return {"bytes": 2 * n + 8 * hidden + 4 * t, "flops": 10.0 * t * (hidden + heads * c["context"] + wide)}
    if kind == "encoder_mlp":
        n = c["batch"] * c["frames"] * c["width"]
        return {"bytes": 4.0 * (4 * 4 * n + 2 * n + 6 * c["width"]), "flops": 12.0 * 4 * n}
    if kind == "encoder_attention":
        n, q = c["batch"] * c["heads"] * c["frames"] ** 2, c["batch"] * c["heads"] * c["frames"] * 64
        return {"bytes": 4.0 * (2 * n + 4 * q), "flops": 4.0 * n}
    if kind == "norm":
        n = c["rows"] * c["cols"]
        return {"bytes": e * (2.0 * n + (2 if c["norm"] == "layer" else 1) * c["cols"]), "flops": 6.0 * n}
    if kind == "prefill":
        t = c["tokens"]
        n = 2 * t * hidden + 2 * heads * t * dim + 2 * heads * t * t + t * t + 3 * t * wide + 3 * t * hidden
        return {"bytes": e * float(n) + 4 * hidden, "flops": 5.0 * heads * t * t + 10.0 * t * wide}
    if kind == "scores":
        n, m = c["heads"] * c["queries"] * c["keys"], c["queries"] * c["keys"] if c["mask"] else 0
        return {"bytes": e * (2.0 * n + m), "flops": 5.0 * n}
    if kind == "keys":
        row = c["batch"] * c["heads"] * c["dim"]
        new, old = row * c["tokens"], row * c["past"]
        return {"bytes": e * float(2 * new + 2 * new + (3 * new + 2 * old) + 2 * (new + old)), "flops": 6.0 * new}
    n = c["batch"] * c["channels"] * c["length"]
    return {"bytes": e * (2.0 * n + 2 * c["channels"]), "flops": 8.0 * n}


def tolerance(case):
    """The 16-bit norms and softmax follow the reference's order of operations to the bit, and so do RoPE and everything that
    only moves data: exact.  Elsewhere about four times what the path showed against the same formulas in f64: one f32 rounding
    here and there, and after a rounding to 16 bits the odd neighbour (one step is 2^-10 of an f16 and 2^-7 of a bf16 value)."""
    kind, d = case["kind"], case.get("dtype", "f32")
    if kind in ("norm", "scores", "keys"):
        return "exact"
    if kind in ("decode", "graph", "prefill"):
        return {"rel": 8e-4, "max": 1.6e-2} if d == "bf16" else {"rel": 1e-4, "max": 2e-3}
    if kind == "group_norm" and d == "f16":
        return {"rel": 5e-5, "max": 2e-3}
    return {"rel": 8e-7, "max": 4e-6}
