"""The work that a user of this package has it do, as cases that can be timed
and checked: ternary Dense layers and SwiGLU FFNs over one row to a whole
prefill, decoder blocks, greedy generation, the fp32 LM head, and a layer
called through the vendor plugin on host buffers.

Sizes are those of the BitNet-2B shape that bench.py measures (hidden 2560,
20 query and 5 key/value heads of 128, FFN 6912, vocab 128256), of the tests,
or generic.  Weights are random ternary codes (P(0) = 1/2), activations
standard normal, norm gains near 1.

`exact` restates each layer in torch at 64 bits: the int8 quantization and the
fp32 roundings between stages belong to the layer's definition (the values
cached or handed from one stage to the next are fp32), every product and sum
is fp64.
"""
import math

import numpy as np
import torch

from loom_amd import accel, bitnet, transformer

SHAPE_2B = dict(hidden=2560, heads=20, kv_heads=5, head_dim=128, inter=6912, theta=500000.0)
SHAPE_SMALL = dict(hidden=1024, heads=16, kv_heads=4, head_dim=64, inter=2816, theta=10000.0)
SHAPES = {"2b": SHAPE_2B, "small": SHAPE_SMALL}
EPS = 1e-5
ACT = {"linear": -1, "relu": 0, "silu": 1, "relu2": 6}


def listed():
    return [
        # one token through one projection: the smallest call a decode loop
        # makes, where the call itself and one launch are what counts
        dict(name="dense_row", kind="dense", m=1, k=2560, n=6912, act="linear", residual=False),
        # a short batch through an ordinary layer of ragged width
        dict(name="dense_ragged", kind="dense", m=37, k=1000, n=777, act="silu", residual=False),
        # the down projection of a 512-token prompt, added to the residual stream
        dict(name="dense_prompt", kind="dense", m=512, k=6912, n=2560, act="linear", residual=True),
        # the up projection of a long prefill
        dict(name="dense_prefill", kind="dense", m=4096, k=2560, n=6912, act="linear", residual=False),
        # the FFN of one decode token, in the default summation order
        dict(name="ffn_row", kind="ffn", m=1, shape="2b", act="silu", norm="strict", bias=False, residual=False),
        # the FFN of a ragged batch, squared-ReLU gate, biases and residual
        dict(name="ffn_batch", kind="ffn", m=300, shape="2b", act="relu2", norm="fast", bias=True, residual=True),
        # one decoder block over a 512-token prompt, default order
        dict(name="block_prompt", kind="block", batch=1, seq=512, shape="2b", norm="strict"),
        # one decoder block over a batch of long prompts
        dict(name="block_prefill", kind="block", batch=8, seq=2048, shape="2b", norm="fast"),
        # greedy generation after a long prompt, whole model
        dict(name="generate", kind="model", batch=1, prompt=2048, steps=64, layers=30, vocab=128256, shape="2b",
             norm="fast"),
        # greedy generation of several sequences at once, default order, a
        # model of fewer layers and a smaller vocabulary
        dict(name="generate_batch", kind="model", batch=8, prompt=120, steps=32, layers=10, vocab=32000, shape="2b",
             norm="strict"),
        # logits and greedy picks of several rows (scoring) over the full vocabulary
        dict(name="head_rows", kind="head", rows=16, vocab=128256, hidden=2560, sequential=False),
        # an FFN layer behind the vendor plugin: host rows in, host rows out
        dict(name="plugin_ffn", kind="plugin", m=8, shape="2b", norm="strict"),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["dense", "dense", "dense", "ffn", "ffn", "block", "block", "model", "head", "plugin"])
    if kind == "dense":
        if rng.random() < 0.6:
            k, n = rng.choice([(2560, 6912), (6912, 2560), (2560, 2560), (2560, 3840), (2560, 640)])
        else:
            k, n = rng.randint(100, 6912), rng.randint(64, 6912)
        return dict(kind=kind, m=_log(rng, 1, 4096), k=k, n=n, act=rng.choice(["linear", "linear", "silu", "relu2"]),
                    residual=rng.random() < 0.4)
    if kind == "ffn":
        return dict(kind=kind, m=_log(rng, 1, 2048), shape=rng.choice(["2b", "2b", "small"]),
                    act=rng.choice(["silu", "relu2"]), norm=rng.choice(["strict", "fast"]), bias=rng.random() < 0.4,
                    residual=rng.random() < 0.4)
    if kind == "block":
        batch = rng.choice([1, 1, 2, 4, 8])
        return dict(kind=kind, batch=batch, seq=_log(rng, 2, 2048), shape=rng.choice(["2b", "2b", "small"]),
                    norm="fast" if batch > 4 else rng.choice(["strict", "fast"]))
    if kind == "model":
        return dict(kind=kind, batch=rng.choice([1, 1, 2, 3, 8]), prompt=_log(rng, 2, 600), steps=_log(rng, 4, 40),
                    layers=rng.randint(2, 8), vocab=_log(rng, 2000, 32000), shape=rng.choice(["2b", "small"]),
                    norm=rng.choice(["strict", "fast"]))
    if kind == "head":
        return dict(kind=kind, rows=_log(rng, 1, 32), vocab=_log(rng, 2000, 128256),
                    hidden=rng.choice([2560, 1024, rng.randint(300, 2560)]), sequential=rng.random() < 0.3)
    return dict(kind=kind, m=_log(rng, 1, 128), shape=rng.choice(["2b", "small"]), norm=rng.choice(["strict", "fast"]))


# ---- inputs, from the seed alone ----------------------------------------------

def _words(rng, rows, cols):
    """Row-major ternary words (16 codes of 2 bits, 0/1/2 = -1/0/+1), P(0) = 1/2."""
    rw = (cols + 15) // 16
    w = rng.integers(0, 1 << 32, size=rows * rw, dtype=np.uint32)
    lo = w & np.uint32(0x55555555)
    hi = (w >> np.uint32(1)) & np.uint32(0x55555555)
    code = ((hi & ~lo) << np.uint32(1)) | (hi ^ np.uint32(0x55555555))
    if cols % 16:
        code.reshape(rows, rw)[:, -1] &= np.uint32((1 << (2 * (cols % 16))) - 1)
    return code


def _matrix(rng, rows, cols):
    return _words(rng, rows, cols), rows, cols, float(np.float32(rng.uniform(0.01, 0.03)))


def _normal(seed, *shape, std=1.0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * std


def _gain(rng, n):
    return rng.uniform(0.5, 1.5, n).astype(np.float32)


def _layer(rng, c):
    """Matrices and gains of one decoder block."""
    h, q, kv, f = c["hidden"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"], c["inter"]
    mats = {name: _matrix(rng, r, k) for name, r, k in
            (("q", q, h), ("k", kv, h), ("v", kv, h), ("o", h, q), ("gate", f, h), ("up", f, h), ("down", h, f))}
    gains = dict(norm1=_gain(rng, h), norm2=_gain(rng, h), attn_inner_norm=_gain(rng, q), ffn_inner_norm=_gain(rng, f))
    return mats, gains


def _load(m):
    return bitnet.TernaryMatrix.from_words(m[0], m[1], m[2], m[3])


def _host(case, seed):
    """Everything of a case that comes from the seed and is not yet on the device."""
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "dense":
        return dict(w=_matrix(rng, case["n"], case["k"]))
    if kind in ("ffn", "plugin"):
        c = SHAPES[case["shape"]]
        h, f = c["hidden"], c["inter"]
        d = dict(gate=_matrix(rng, f, h), up=_matrix(rng, f, h), down=_matrix(rng, h, f), inner=_gain(rng, f))
        if case.get("bias"):
            d["bias"] = rng.standard_normal(2 * f + h, dtype=np.float32) * np.float32(0.5)
        if kind == "plugin":
            d["x"] = rng.standard_normal((case["m"], h), dtype=np.float32)
        return d
    if kind == "block":
        return dict(layer=_layer(rng, SHAPES[case["shape"]]))
    if kind == "model":
        c = SHAPES[case["shape"]]
        return dict(layers=[_layer(rng, c) for _ in range(min(4, case["layers"]))], final=_gain(rng, c["hidden"]),
                    ids=rng.integers(0, case["vocab"], (case["batch"], case["prompt"])).astype(np.int32))
    return {}


def _even(n):
    return n + n % 2  # the strict prefill takes an even number of cached rows


def _config(c, norm, msl, batch):
    return transformer.BlockConfig(c["hidden"], c["heads"], c["kv_heads"], c["head_dim"], c["inter"], max_seq_len=msl,
                                   max_batch=batch, rope_theta=c["theta"], norm_eps=EPS, ffn_activation=ACT["silu"],
                                   norm=norm)


def _weights(layer):
    mats, gains = layer
    return transformer.BlockWeights(**{k: _load(m) for k, m in mats.items()}, **gains)


def _blob(m):
    """A BITNET_TERNARY entity blob: rows, cols, offset, scale, words per row, words."""
    words, rows, cols, scale = m
    head = np.array([rows, cols, 0, 0, (cols + 15) // 16, words.size], np.uint32)
    head[3:4] = np.array([scale], np.float32).view(np.uint32)
    return head.tobytes() + words.tobytes()


def prepare(case, seed):
    kind = case["kind"]
    d = _host(case, seed)
    s = dict(case=case)
    if kind == "dense":
        s["w"] = _load(d["w"])
        s["x"] = _normal(seed, case["m"], case["k"])
        s["residual"] = _normal(seed + 1, case["m"], case["n"]) if case["residual"] else None
    elif kind == "ffn":
        h = SHAPES[case["shape"]]["hidden"]
        s.update(gate=_load(d["gate"]), up=_load(d["up"]), down=_load(d["down"]))
        s["inner"] = torch.from_numpy(d["inner"]).cuda()
        s["bias"] = torch.from_numpy(d["bias"]).cuda() if case["bias"] else None
        s["x"] = _normal(seed, case["m"], h)
        s["residual"] = _normal(seed + 1, case["m"], h) if case["residual"] else None
    elif kind == "block":
        c = SHAPES[case["shape"]]
        s["block"] = transformer.BitNetBlock(_config(c, case["norm"], _even(case["seq"]), case["batch"]),
                                             _weights(d["layer"]))
        s["x"] = _normal(seed, case["batch"], case["seq"], c["hidden"])
    elif kind == "model":
        # more layers than four repeat the four sets of weights (every layer
        # holds a copy of its own on the device)
        c = SHAPES[case["shape"]]
        total = case["prompt"] + case["steps"]
        four = [_weights(layer) for layer in d["layers"]]
        emb = _normal(seed, case["vocab"], c["hidden"], std=0.02).cpu().numpy()
        s["model"] = transformer.Transformer(
            _config(c, case["norm"], _even(total), case["batch"]), [four[i % len(four)] for i in range(case["layers"])], emb,
            d["final"], vocab=case["vocab"], final_norm_eps=EPS, max_tokens=total + 1, max_prefill=case["prompt"])
        s["ids"] = d["ids"]
    elif kind == "head":
        s["table"] = _normal(seed, case["vocab"], case["hidden"], std=0.02)
        s["x"] = _normal(seed + 1, case["rows"], case["hidden"])
    else:
        c = SHAPES[case["shape"]]
        s["plugin"] = accel.open_amd()
        desc = accel.LayerDesc("BitNetSwiGLU", "TERNARY", "m=%d,k=%d,n=%d,act=1,norm=%s"
                               % (case["m"], c["hidden"], c["inter"], case["norm"]))
        blob = _blob(d["gate"]) + _blob(d["up"]) + _blob(d["down"]) + d["inner"].tobytes()
        s["layer"] = s["plugin"].compile_layer(desc, blob).layer
        s["x"] = d["x"]
        s["out"] = np.empty((case["m"], c["hidden"]), np.float32)
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "dense":
        pre, post = bitnet.dense_forward_packed_ternary(state["w"], state["x"], ACT[case["act"]],
                                                        residual=state["residual"])
        return (pre,) if post is pre else (pre, post)
    if kind == "ffn":
        return bitnet.swiglu_forward_packed_ternary(state["gate"], state["up"], state["down"], state["x"],
                                                    state["inner"], EPS, ACT[case["act"]], case["norm"], state["bias"],
                                                    state["residual"])
    if kind == "block":
        # the block works in place on the residual stream, which a model hands
        # it anew with every prompt
        x, _ = state["block"].forward(state["x"].clone())
        return x
    if kind == "model":
        model = state["model"]
        model.prefill(state["ids"])
        logits = model.decode(case["steps"], logits=True)
        return {"logits": logits, "tokens": model.tokens()}
    if kind == "head":
        logits = transformer.lm_head(state["table"], state["x"], case["sequential"])
        return {"logits": logits, "ids": transformer.greedy_sample(logits)}
    state["layer"].infer(state["x"], state["out"])
    return state["out"]


# ---- what a pass cannot do without --------------------------------------------

def _mat(rows, cols):
    return rows * ((cols + 15) // 16) * 4


def _layer_bytes(c):
    h, q, kv, f = c["hidden"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"], c["inter"]
    return _mat(q + 2 * kv, h) + _mat(h, q) + 2 * _mat(f, h) + _mat(h, f) + 4 * (2 * h + q + f)


def _layer_flops(c, rows):
    h, q, kv, f = c["hidden"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"], c["inter"]
    return 2.0 * rows * (h * (q + 2 * kv) + q * h + 3 * h * f)


def work(case):
    kind = case["kind"]
    if kind == "dense":
        m, k, n = case["m"], case["k"], case["n"]
        outs = 2 if case["act"] != "linear" else 1
        return {"bytes": _mat(n, k) + 4 * m * (k + n * (outs + case["residual"])), "flops": 2.0 * m * k * n}
    if kind in ("ffn", "plugin"):
        c = SHAPES[case["shape"]]
        h, f, m = c["hidden"], c["inter"], case["m"]
        by = 2 * _mat(f, h) + _mat(h, f) + 4 * f + 8 * m * h
        if kind == "ffn":
            by += 4 * m * f + (4 * (2 * f + h) if case["bias"] else 0) + (4 * m * h if case["residual"] else 0)
        return {"bytes": by, "flops": 6.0 * m * h * f}
    if kind == "block":
        c = SHAPES[case["shape"]]
        b, s = case["batch"], case["seq"]
        kv = c["kv_heads"] * c["head_dim"]
        attn = 4.0 * b * c["heads"] * c["head_dim"] * s * (s + 1) / 2
        return {"bytes": _layer_bytes(c) + 4 * b * s * (2 * c["hidden"] + 2 * kv),
                "flops": _layer_flops(c, b * s) + attn}
    if kind == "model":
        # weights once in the prefill and once a step; each step the cached
        # rows and the table's entries at one byte (the greedy pick needs no
        # more of most rows) and, once, the logits asked for
        c = SHAPES[case["shape"]]
        b, p, t, n, v = case["batch"], case["prompt"], case["steps"], case["layers"], case["vocab"]
        h, kv = c["hidden"], c["kv_heads"] * c["head_dim"]
        cached = sum(2 * kv * 4 * b * (p + i) for i in range(t))
        by = (t + 1) * (n * _layer_bytes(c) + v * h) + n * cached + n * 8 * b * p * kv + 4 * v * (h + b)
        attn = 4.0 * b * c["heads"] * c["head_dim"] * (p * (p + 1) / 2 + sum(p + i + 1 for i in range(t)))
        return {"bytes": by, "flops": n * (_layer_flops(c, b * (p + t)) + attn) + 2.0 * b * (t + 2) * v * h}
    r, v, h = case["rows"], case["vocab"], case["hidden"]
    return {"bytes": 4 * (v * h + r * h + r * v), "flops": 2.0 * r * v * h}


def tolerance(case):
    # Measured: the strict and the fast summation order of every kind give the
    # same bits on these inputs, or an fp32 rounding apart; against `exact`
    # the differences are the roundings of fp32 results.
    kind = case["kind"]
    if kind == "head":
        return {"rel": 1e-7, "max": 2.5e-7, "differ": 0.01}  # seen: 2.5e-8, 6e-8 (fp32 of an fp64 sum)
    if kind == "dense":
        return {"rel": 2.6e-7, "max": 1.1e-6}  # seen: 6.5e-8, 2.7e-7 (residual, then the activation's product)
    if kind == "model":
        # a normalized value one fp32 ulp off moves an int8 code by one now
        # and then, which the layers after it carry on
        return {"rel": 1e-3, "max": 0.05, "differ": 0.01}
    # roundings of the output (seen: 3e-8), and one moved int8 code in some
    # hundred rows: 5e-6 in one of 2048 rows was seen for a scale one fp64 ulp off
    return {"rel": 2e-5, "max": 0.02}


# ---- the same in torch at 64 bits -----------------------------------------------

def _codes(m):
    """The ternary weights as fp64 (rows, cols) on the device."""
    words, rows, cols, _ = m
    w = torch.from_numpy(words.view(np.int32).reshape(rows, -1)).cuda()
    t = torch.stack([(w >> (2 * i)) & 3 for i in range(16)], dim=2).reshape(rows, -1)[:, :cols]
    return t.to(torch.float64) - 1.0


def _quant(x):
    """Per row: int8 values (as fp64) and the fp32 absolute maximum, at least 1e-5."""
    x = x.double()
    amax = x.abs().amax(1).float().clamp_min(1e-5).double()
    p = x * torch.full_like(amax, 127.0).div_(amax)[:, None]  # (127.0 / amax is a reciprocal and a product)
    q = torch.sign(p) * torch.floor(p.abs() + 0.5)
    return q.clamp_(-128, 127), amax


def _ternary(q, amax, m):
    out = torch.empty(q.shape[0], m[1], dtype=torch.float64, device="cuda")
    w = _codes(m).t().contiguous()
    for i in range(0, q.shape[0], 4096):
        out[i:i + 4096] = q[i:i + 4096] @ w
    scale = float(np.float32(m[3])) * amax / 127.0
    return out * scale[:, None]


def _rms(x, eps=EPS):
    return torch.sqrt(x.double().square().mean(1) + eps)[:, None]


def _gate(g, u, act):
    if act == "relu2":
        return g.clamp_min(0).square() * u
    return g * torch.sigmoid(g) * u


def _ffn(x, d, act, bias=None):
    """(normalized h, output) of a SwiGLU FFN, both fp32 as they are handed on."""
    f = d["gate"][1]
    q, amax = _quant(x)
    g, u = _ternary(q, amax, d["gate"]), _ternary(q, amax, d["up"])
    if bias is not None:
        g, u = g + bias[:f], u + bias[f:2 * f]
    h = _gate(g, u, act).float()
    h = (h.double() / _rms(h) * torch.from_numpy(d["inner"]).cuda().double()).float()
    q, amax = _quant(h)
    o = _ternary(q, amax, d["down"])
    return h, (o if bias is None else o + bias[2 * f:]).float()


def _rope(x, heads, hd, theta, seq):
    """Rotates (batch * seq, heads * hd) fp64 rows by their positions."""
    half = hd // 2
    pos = torch.arange(seq, dtype=torch.float64, device="cuda").repeat(x.shape[0] // seq)
    inv = torch.tensor(theta, dtype=torch.float64, device="cuda") ** (
        torch.arange(half, dtype=torch.float64, device="cuda") * 2 / hd)
    a = pos[:, None] / inv[None]
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    v = x.reshape(x.shape[0], heads, hd)
    lo, hi = v[..., :half], v[..., half:]
    return torch.cat([lo * c - hi * s, lo * s + hi * c], -1).reshape(x.shape)


def _attention(q, k, v, c, batch, seq):
    hd, group = c["head_dim"], c["heads"] // c["kv_heads"]
    out = torch.empty_like(q)
    late = torch.ones(seq, seq, dtype=torch.bool, device="cuda").triu(1)
    for b in range(batch):
        r = slice(b * seq, (b + 1) * seq)
        for h in range(c["heads"]):
            cq = slice(h * hd, (h + 1) * hd)
            ck = slice(h // group * hd, (h // group + 1) * hd)
            sc = (q[r, cq] @ k[r, ck].double().t().contiguous() / math.sqrt(hd)).masked_fill_(late, -math.inf)
            p = torch.exp(sc - sc.amax(1, keepdim=True))  # (torch's fp64 softmax over long rows is off by 4e-8)
            out[r, cq] = p @ v[r, ck].double() / p.sum(1, keepdim=True)
    return out


def _block(x, layer, c, batch, seq):
    mats, gains = layer
    g = {k: torch.from_numpy(a).cuda().double() for k, a in gains.items()}
    q, amax = _quant((x.double() / _rms(x) * g["norm1"]).float())
    k = _ternary(q, amax, mats["k"]).float()
    v = _ternary(q, amax, mats["v"]).float()
    k = _rope(k.double(), c["kv_heads"], c["head_dim"], c["theta"], seq).float()
    a = _attention(_rope(_ternary(q, amax, mats["q"]), c["heads"], c["head_dim"], c["theta"], seq), k, v, c, batch, seq)
    q, amax = _quant(a / _rms(a) * g["attn_inner_norm"])
    x = _ternary(q, amax, mats["o"]).float() + x
    y = (x.double() / _rms(x) * g["norm2"]).float()
    d = dict(gate=mats["gate"], up=mats["up"], down=mats["down"], inner=gains["ffn_inner_norm"])
    return _ffn(y, d, "silu")[1] + x


def exact(case, seed):
    kind = case["kind"]
    d = _host(case, seed)
    if kind == "dense":
        q, amax = _quant(_normal(seed, case["m"], case["k"]))
        v = _ternary(q, amax, d["w"])
        if case["residual"]:
            v = v + _normal(seed + 1, case["m"], case["n"]).double()
        if case["act"] == "linear":
            return (v,)
        return (v, v * torch.sigmoid(v) if case["act"] == "silu" else v.clamp_min(0).square())
    if kind == "ffn":
        x = _normal(seed, case["m"], SHAPES[case["shape"]]["hidden"])
        bias = torch.from_numpy(d["bias"]).cuda().double() if case["bias"] else None
        h, o = _ffn(x, d, case["act"], bias)
        if case["residual"]:
            o = o.double() + _normal(seed + 1, *x.shape).double()
        return h.double(), o.double()
    if kind == "block":
        c = SHAPES[case["shape"]]
        x = _normal(seed, case["batch"] * case["seq"], c["hidden"])
        y = _block(x, d["layer"], c, case["batch"], case["seq"])
        return y.double().reshape(case["batch"], case["seq"], -1)
    if kind == "model":
        # a chain of greedy picks and int8 roundings has no 64-bit value of
        # its own: the blocks and the head are checked by themselves
        return None
    if kind == "head":
        table, x = _normal(seed, case["vocab"], case["hidden"], std=0.02), _normal(seed + 1, case["rows"], case["hidden"])
        logits = torch.empty(case["rows"], case["vocab"], dtype=torch.float64, device="cuda")
        for i in range(0, case["vocab"], 16384):
            logits[:, i:i + 16384] = x.double() @ table[i:i + 16384].double().t().contiguous()
        return {"logits": logits, "ids": None}
    return _ffn(torch.from_numpy(d["x"]).cuda(), d, "silu")[1].double().cpu().numpy()
