"""Performance cases: what a program that uses this framework has it do.

Each case is one pass through a public entry point at a size that is used:
the standalone operators on device buffers (quantised and fp32 matvec, fp32
matmul), two decoded tokens and whole prompts (and the token that follows
them, which reads the cache they wrote) through quantised models with their
logits, whole generate calls (greedy and sampled), and the fp32 model path.
The shapes are the repository's synthetic workloads: the TinyLlama shape, the
Llama-2-7B widths and the small test shapes. ``listed`` names twelve of them,
``draw`` makes more of the same kinds over the whole ranges.

Inputs come from the seed alone (torch's generator on the GPU): N(0, 0.02)
weights quantised in blocks, norms around one, uniform token ids, and K/V
rows with the spread that such weights give.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import nutllm_amd as nut

SHAPES = {
    "tiny": dict(layers=2, heads=4, dim=64, head_dim=16, ffn_dim=172, vocab_size=256,
                 kv_heads=2),
    "step_gqa2": dict(layers=2, heads=4, dim=256, head_dim=64, ffn_dim=512, vocab_size=512,
                      kv_heads=2),
    "step_gqa4": dict(layers=2, heads=8, dim=512, head_dim=64, ffn_dim=768, vocab_size=512,
                      kv_heads=2),
    "step_mha128": dict(layers=2, heads=2, dim=256, head_dim=128, ffn_dim=512, vocab_size=512,
                        kv_heads=2),
    "tinyllama": dict(layers=22, heads=32, dim=2048, head_dim=64, ffn_dim=5632,
                      vocab_size=32000, kv_heads=4),
    "llama7b": dict(layers=2, heads=32, dim=4096, head_dim=128, ffn_dim=11008,
                    vocab_size=32000, kv_heads=32),
}
EOS = 1
MAX_SEQ = 2176
SIGMA = 0.02
INT8, INT4 = "int8", "int4"


def listed():
    return [
        # the smallest calls: the key and value projections of one TinyLlama
        # layer, two matrices over one input
        dict(name="matvec_int8_small", kind="matvec_q", rows=256, cols=2048, type=INT8, block=32),
        # the gate and up projections of one Llama-2-7B layer
        dict(name="matvec_int4_large", kind="matvec_q", rows=11008, cols=4096, type=INT4,
             block=32),
        # a classifier: fp32 logits of one hidden state
        dict(name="matvec_f32_head", kind="matvec_f32", rows=32000, cols=2048),
        # the reference's own GEMM benchmark
        dict(name="matmul_f32_768", kind="matmul_f32", m=768, k=768, n=768),
        # a GEMM of sizes that no tile divides
        dict(name="matmul_f32_ragged", kind="matmul_f32", m=1000, k=2047, n=1531),
        # two tokens of a serving loop that samples by itself, deep in a context
        dict(name="decode_int8_2k", kind="decode", shape="tinyllama", layers=22, type=INT8,
             block=32, context=2050),
        # a chat turn's whole greedy continuation of a short prompt
        dict(name="generate_greedy_int4", kind="generate", shape="tinyllama", layers=22,
             type=INT4, prompt=5, tokens=16, temperature=0.0, top_p=1.0),
        # the same with temperature and nucleus sampling
        dict(name="generate_sampled_int4", kind="generate", shape="tinyllama", layers=22,
             type=INT4, prompt=20, tokens=16, temperature=0.8, top_p=0.9),
        # a long document read before the first answer tokens
        dict(name="prefill_int8_2048", kind="prefill", shape="tinyllama", layers=22, type=INT8,
             block=32, tokens=2048),
        # two layers of the 7B widths over an ordinary, odd prompt
        dict(name="prefill_7b_int4_301", kind="prefill", shape="llama7b", layers=2, type=INT4,
             block=32, tokens=301),
        # fp32 layers over an ordinary prompt, every row's hidden state
        dict(name="prefill_f32_301", kind="prefill_f32", shape="tinyllama", layers=4, tokens=301),
        # two tokens through fp32 layers, in an ordinary context
        dict(name="decode_f32_700", kind="decode_f32", shape="tinyllama", layers=4, context=700),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _layers(rng, shape, most):
    return rng.randint(1, most) if shape == "tinyllama" else SHAPES[shape]["layers"]


def draw(rng):
    kind = rng.choice(["matvec_q", "matvec_q", "matvec_f32", "matmul_f32", "matmul_f32", "decode",
                       "decode", "generate", "prefill", "prefill", "prefill_f32", "decode_f32"])
    qtype = rng.choice([INT8, INT4])
    if kind == "matvec_q":
        cols = _log_int(rng, 64, 11008)
        if rng.random() < 0.6:  # whole blocks along the rows, as every model has them
            cols = max(32, cols // 32 * 32)
        return dict(kind=kind, rows=_log_int(rng, 64, 16384), cols=cols, type=qtype,
                    block=rng.choice([32, 32, 32, 64]))
    if kind == "matvec_f32":
        return dict(kind=kind, rows=_log_int(rng, 256, 32000), cols=_log_int(rng, 64, 8192))
    if kind == "matmul_f32":
        m, k, n = (_log_int(rng, 24, 4096) for _ in range(3))
        if rng.random() < 0.4:  # a model's widths
            k, n = max(64, k // 64 * 64), max(64, n // 64 * 64)
        return dict(kind=kind, m=m, k=k, n=n)
    if kind == "generate":
        sampled = rng.random() < 0.5
        return dict(kind=kind, shape="tinyllama", layers=rng.randint(2, 22), type=qtype,
                    prompt=_log_int(rng, 1, 300), tokens=_log_int(rng, 4, 32),
                    temperature=round(rng.uniform(0.5, 1.1), 3) if sampled else 0.0,
                    top_p=round(rng.uniform(0.7, 1.0), 3) if sampled else 1.0)
    shape = rng.choice(["tinyllama", "tinyllama", "tinyllama", "llama7b", "llama7b", "tiny",
                        "step_gqa2", "step_gqa4", "step_mha128"])
    if kind == "decode":
        return dict(kind=kind, shape=shape, layers=_layers(rng, shape, 22), type=qtype,
                    block=rng.choice([32, 32, 32, 64]), context=_log_int(rng, 1, 2100))
    if kind == "prefill":
        return dict(kind=kind, shape=shape, layers=_layers(rng, shape, 12), type=qtype,
                    block=32, tokens=_log_int(rng, 1, 2048))
    if kind == "prefill_f32":
        return dict(kind=kind, shape=shape, layers=_layers(rng, shape, 4),
                    tokens=_log_int(rng, 1, 300))
    return dict(kind=kind, shape=shape, layers=_layers(rng, shape, 4),
                context=_log_int(rng, 1, 2100))


# ------------------------------------------------------------------ inputs --

def _gen(seed, stream):
    return torch.Generator(device="cuda").manual_seed(seed * 1000003 + stream)


def _normal(seed, stream, *shape, sigma=1.0):
    return torch.randn(*shape, generator=_gen(seed, stream), device="cuda") * sigma


def _tokens(seed, stream, vocab, count):
    t = torch.randint(2, vocab, (count,), generator=_gen(seed, stream), device="cuda")
    return t.cpu().numpy().astype(np.int32)


def _quantised(w, qtype, block):
    """Codes and scale of symmetric blocks along the flattened matrix."""
    flat = w.reshape(-1)
    pad = -flat.numel() % block
    b = torch.nn.functional.pad(flat, (0, pad)).reshape(-1, block)
    top = 7 if qtype == INT4 else 127
    scale = (b.abs().amax(1) / top).half()
    inv = torch.where(scale > 0, 1.0 / scale.float(), torch.zeros_like(scale, dtype=torch.float32))
    codes = (b * inv[:, None]).round_().clamp_(-top, top).to(torch.int8)
    return codes, scale


def _stored(codes, scale, count, qtype):
    """The reference's storage: bytes or nibbles, fp16 scale bits."""
    flat = codes.reshape(-1)[:count]
    if qtype == INT4:
        flat = torch.nn.functional.pad(flat, (0, count & 1)).reshape(-1, 2)
        data = (flat[:, 0] & 15) | ((flat[:, 1] & 15) << 4)
    else:
        data = flat
    return (data.contiguous().view(torch.uint8).cpu().numpy(),
            scale.view(torch.int16).cpu().numpy().view(np.uint16))


def _dense(codes, scale, rows, cols):
    return (codes.double() * scale.double()[:, None]).reshape(-1)[:rows * cols].reshape(rows, cols)


def _config(case):
    return nut.Config(**{**SHAPES[case["shape"]], "layers": case["layers"]}, max_seq=MAX_SEQ,
                      eos_token=EOS)


def _shape(case):
    s = dict(SHAPES[case["shape"]], layers=case["layers"])
    s["kv_dim"] = s["kv_heads"] * s["head_dim"]
    return s


def _projections(s):
    """[out x in] of a layer's projections, in the order of PROJECTIONS."""
    d, f, kv = s["dim"], s["ffn_dim"], s["kv_dim"]
    return dict(query=(d, d), key=(kv, d), value=(kv, d), output=(d, d), gate=(f, d), up=(f, d),
                down=(d, f))


def _weight(seed, layer, index, rows, cols):
    return _normal(seed, 100 + 16 * layer + index, rows, cols, sigma=SIGMA)


def _norm(seed, stream, dim):
    return 1.0 + _normal(seed, stream, dim, sigma=0.1)


def _norms(seed, layer, dim):
    return (_norm(seed, 100 + 16 * layer + 8, dim), _norm(seed, 100 + 16 * layer + 9, dim))


def _globals(case, seed):
    s = _shape(case)
    # a trained head's logits spread over several units, which is what the
    # sampler's nucleus depends on
    spread = 0.06 if case["kind"] == "generate" else SIGMA
    return (_normal(seed, 1, s["vocab_size"], s["dim"], sigma=SIGMA),
            _norm(seed, 2, s["dim"]), _normal(seed, 3, s["vocab_size"], s["dim"], sigma=spread))


def _host(t):
    return t.cpu().numpy()


def _model(case, seed):
    s, block = _shape(case), case.get("block", 32)
    m = nut.DeviceModel(_config(case), nut.INT4 if case["type"] == INT4 else nut.INT8)
    m.set_globals(*map(_host, _globals(case, seed)))
    for layer in range(s["layers"]):
        mats = {}
        for i, (name, (rows, cols)) in enumerate(_projections(s).items()):
            codes, scale = _quantised(_weight(seed, layer, i, rows, cols), case["type"], block)
            mats[name] = (*_stored(codes, scale, rows * cols, case["type"]), rows, cols, block)
        m.set_layer(layer, mats, *map(_host, _norms(seed, layer, s["dim"])))
    return m


def _fmodel(case, seed):
    s = _shape(case)
    m = nut.DeviceFModel(_config(case), tied=True)
    m.set_globals(*map(_host, _globals(case, seed)[:2]))
    for layer in range(s["layers"]):
        w = {name: _host(_weight(seed, layer, i, cols, rows))  # [in x out]
             for i, (name, (rows, cols)) in enumerate(_projections(s).items())}
        m.set_layer(layer, w, *map(_host, _norms(seed, layer, s["dim"])))
    return m


def _context(case, seed):
    """K and V rows of the positions before the decoded token."""
    s = _shape(case)
    sigma = SIGMA * math.sqrt(s["dim"])
    shape = (s["layers"], s["kv_heads"], case["context"], s["head_dim"])
    return _normal(seed, 5, *shape, sigma=sigma), _normal(seed, 6, *shape, sigma=sigma)


def _next(case, seed, count):
    """The tokens that the caller goes on with."""
    return [int(t) for t in _tokens(seed, 7, _shape(case)["vocab_size"], count)]


class _Buffer:
    """A torch tensor as the device buffer that the operators take."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = ctypes.c_void_p(tensor.data_ptr())


def _matvec_q_inputs(case, seed):
    """Two matrices of one shape, and their input."""
    w = [_normal(seed, 10 + i, case["rows"], case["cols"], sigma=SIGMA) for i in range(2)]
    return ([_quantised(a, case["type"], case["block"]) for a in w],
            _normal(seed, 2, case["cols"]))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "matvec_q":
        rows, cols = case["rows"], case["cols"]
        matrices, x = _matvec_q_inputs(case, seed)
        qtype = nut.INT4 if case["type"] == INT4 else nut.INT8
        w = [nut.QWeight(*_stored(codes, scale, rows * cols, case["type"]), rows, cols, qtype,
                         case["block"]) for codes, scale in matrices]
        return dict(kind=kind, w=w, x=_Buffer(x),
                    y=[_Buffer(torch.empty(rows, device="cuda")) for _ in w])
    if kind == "matvec_f32":
        w = _normal(seed, 1, case["rows"], case["cols"], sigma=SIGMA)
        x, y = _normal(seed, 2, case["cols"]), torch.empty(case["rows"], device="cuda")
        return dict(kind=kind, keep=(w, x), y=y, lib=nut.lib(),
                    args=(w.data_ptr(), case["rows"], case["cols"], x.data_ptr(), y.data_ptr(),
                          None))
    if kind == "matmul_f32":
        m, k, n = case["m"], case["k"], case["n"]
        a, b = _normal(seed, 1, m, k), _normal(seed, 2, k, n)
        c = torch.empty(m, n, device="cuda")
        return dict(kind=kind, keep=(a, b), c=c, lib=nut.lib(),
                    args=(a.data_ptr(), b.data_ptr(), c.data_ptr(), m, k, n, None))
    s = _shape(case)
    state = dict(kind=kind, cache=nut.KVCache(_config(case)))
    state["model"] = _fmodel(case, seed) if kind.endswith("_f32") else _model(case, seed)
    if kind.startswith("decode"):
        state["next"] = _next(case, seed, 2)
        state["context"] = case["context"]
        state["cache"].write_positions(0, *map(_host, _context(case, seed)))
    elif kind == "generate":
        state["prompt"] = _tokens(seed, 4, s["vocab_size"], case["prompt"])
        state["how"] = (case["tokens"], case["temperature"], case["top_p"], seed & 0x7fffffff)
    else:
        state["tokens"] = _tokens(seed, 4, s["vocab_size"], case["tokens"])
        state["next"] = _next(case, seed, 1)
    return state


# --------------------------------------------------------------------- run --

def run(state):
    kind = state["kind"]
    if kind == "matvec_q":
        for w, y in zip(state["w"], state["y"]):
            w.matvec(state["x"], y)
        return [y.tensor for y in state["y"]]
    if kind == "matvec_f32":
        nut.check(state["lib"].nut_matvec_f32(*state["args"]))
        return state["y"]
    if kind == "matmul_f32":
        nut.check(state["lib"].nut_matmul_f32(*state["args"]))
        return state["c"]
    model, cache = state["model"], state["cache"]
    if kind.startswith("decode"):
        cache.set_length(state["context"])
        steps = []
        for token in state["next"]:
            hidden = model.decode(cache, token)
            steps.append(dict(hidden=hidden))
            if kind == "decode":
                steps[-1]["logits"] = model.logits(hidden)
        return steps
    if kind == "prefill":
        hidden = model.prefill(cache, state["tokens"])
        return dict(hidden=hidden, logits=model.logits(hidden),
                    next=model.decode(cache, state["next"][0]))
    if kind == "prefill_f32":
        rows = model.prefill(cache, state["tokens"])
        return dict(rows=rows, next=model.decode(cache, state["next"][0]))
    # generate: the prompt's own scores, then its continuation
    logits = model.logits(model.prefill(cache, state["prompt"]))
    tokens, temperature, top_p, seed = state["how"]
    if temperature > 0:
        ids, _ = model.generate_sampled(state["prompt"], tokens, temperature, top_p, seed)
    else:
        ids, _ = model.generate(state["prompt"], tokens)
    return dict(ids=np.asarray(ids, np.int32), logits=logits)


# -------------------------------------------------------------------- work --

def _layer_work(case, tokens, context):
    """Bytes and operations of `tokens` new positions after `context`."""
    s = _shape(case)
    weights = sum(r * c for r, c in _projections(s).values())
    if "type" in case:
        block = case.get("block", 32)
        size = weights * (0.5 if case["type"] == INT4 else 1) + 2 * weights / block
    else:
        size = 4 * weights
    seen = tokens * context + tokens * (tokens + 1) / 2  # (query, key) pairs
    kv = 2 * 4 * s["kv_dim"]  # a position's K and V rows
    return dict(bytes=s["layers"] * (size + 8 * s["dim"] + kv * (context + tokens)),
                flops=s["layers"] * (2 * weights * tokens + 4 * seen * s["dim"]))


def _head_work(case):
    s = _shape(case)
    n = s["vocab_size"] * s["dim"]
    return dict(bytes=4 * (n + 2 * s["dim"] + s["vocab_size"]), flops=2 * n)


def _sum(*works):
    return {k: sum(w[k] for w in works) for k in ("bytes", "flops")}


def work(case):
    kind = case["kind"]
    if kind == "matvec_q":
        n = case["rows"] * case["cols"]
        size = n * (0.5 if case["type"] == INT4 else 1) + 2 * n / case["block"]
        return dict(bytes=2 * size + 4 * (2 * case["rows"] + case["cols"]), flops=4 * n)
    if kind == "matvec_f32":
        n = case["rows"] * case["cols"]
        return dict(bytes=4 * (n + case["rows"] + case["cols"]), flops=2 * n)
    if kind == "matmul_f32":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=4 * (m * k + k * n + m * n), flops=2 * m * k * n)
    if kind == "prefill":
        return _sum(_layer_work(case, case["tokens"], 0), _head_work(case),
                    _layer_work(case, 1, case["tokens"]))
    if kind == "prefill_f32":
        return _sum(_layer_work(case, case["tokens"], 0), _layer_work(case, 1, case["tokens"]))
    if kind.startswith("decode"):
        steps = [_layer_work(case, 1, case["context"] + i) for i in range(2)]
        return _sum(*steps, *([_head_work(case)] * 2 if kind == "decode" else []))
    steps = [_sum(_layer_work(case, 1, case["prompt"] + i), _head_work(case))
             for i in range(case["tokens"])]
    prompt = _layer_work(case, case["prompt"], 0)
    return _sum(prompt, prompt, _head_work(case), *steps)


def tolerance(case):
    # about four times the largest error against exact() over the ranges:
    # 3.5e-7 for a row's fp32 sum, 8e-7 for the longer sums of a product,
    # 1.1e-6 through fp32 layers, 3.2e-6 through a whole quantised model
    rel = {"matvec_q": 2e-6, "matvec_f32": 2e-6, "matmul_f32": 5e-6, "decode_f32": 5e-6,
           "prefill_f32": 5e-6}
    return {"rel": rel.get(case["kind"], 1.5e-5)}


# ------------------------------------------------------------------- exact --

def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w


def _rotate(x, first):
    """x [tokens, heads, head_dim]: pairs (2i, 2i + 1) at positions first ..."""
    t, _, hd = x.shape
    pair = torch.arange(hd // 2, device=x.device, dtype=torch.float64)
    pos = torch.arange(first, first + t, device=x.device, dtype=torch.float64)
    angle = pos[:, None] * 10000.0 ** (-2.0 * pair / hd)[None, :]
    cos, sin = torch.cos(angle)[:, None, :], torch.sin(angle)[:, None, :]
    even, odd = x[..., 0::2], x[..., 1::2]
    return torch.stack((even * cos - odd * sin, even * sin + odd * cos), -1).reshape(x.shape)


def _attend(q, k, v, first):
    """Causal attention of one head: q [t, hd] at positions first ..., k and
    v [first + t, hd]."""
    score = q @ k.T.contiguous() / math.sqrt(q.shape[1])
    pos = torch.arange(k.shape[0], device=q.device)
    row = torch.arange(first, first + q.shape[0], device=q.device)
    score = score.masked_fill(pos[None, :] > row[:, None], -math.inf)
    return torch.softmax(score, -1) @ v


def _exact_layers(case, seed, x, past=None):
    """The hidden states after every layer, in 64 bits."""
    s = _shape(case)
    quantised = not case["kind"].endswith("_f32")
    t, heads, kvh, hd = x.shape[0], s["heads"], s["kv_heads"], s["head_dim"]
    first = 0 if past is None else past[0].shape[2]
    for layer in range(s["layers"]):
        w = {}
        for i, (name, (rows, cols)) in enumerate(_projections(s).items()):
            if quantised:
                dense = _weight(seed, layer, i, rows, cols)
                w[name] = _dense(*_quantised(dense, case["type"], case.get("block", 32)), rows,
                                 cols).T
            else:
                w[name] = _weight(seed, layer, i, cols, rows).double()
        attention_norm, ffn_norm = (n.double() for n in _norms(seed, layer, s["dim"]))
        h = _rms(x, attention_norm)
        q = _rotate((h @ w["query"]).reshape(t, heads, hd), first)
        k = _rotate((h @ w["key"]).reshape(t, kvh, hd), first)
        v = (h @ w["value"]).reshape(t, kvh, hd)
        context = []
        for head in range(heads):
            g = head // (heads // kvh)
            kh, vh = k[:, g], v[:, g]
            if past is not None:
                kh = torch.cat((past[0][layer, g].double(), kh))
                vh = torch.cat((past[1][layer, g].double(), vh))
            context.append(_attend(q[:, head].contiguous(), kh.contiguous(), vh.contiguous(),
                                   first))
        x = x + torch.cat(context, 1) @ w["output"]
        h = _rms(x, ffn_norm)
        x = x + (torch.nn.functional.silu(h @ w["gate"]) * (h @ w["up"])) @ w["down"]
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind == "matvec_q":
        matrices, x = _matvec_q_inputs(case, seed)
        return [_dense(*m, case["rows"], case["cols"]) @ x.double() for m in matrices]
    if kind == "matvec_f32":
        return (_normal(seed, 1, case["rows"], case["cols"], sigma=SIGMA).double()
                @ _normal(seed, 2, case["cols"]).double())
    if kind == "matmul_f32":
        return (_normal(seed, 1, case["m"], case["k"]).double()
                @ _normal(seed, 2, case["k"], case["n"]).double())
    s = _shape(case)
    embeddings, final_norm, head = _globals(case, seed)
    past = None
    if kind.startswith("decode"):
        ids, past = _next(case, seed, 2), _context(case, seed)
    elif kind == "generate":
        ids = list(_tokens(seed, 4, s["vocab_size"], case["prompt"]))
    else:
        ids = list(_tokens(seed, 4, s["vocab_size"], case["tokens"])) + _next(case, seed, 1)
    x = embeddings[torch.tensor(np.asarray(ids, np.int64)).cuda()].double()
    x = _exact_layers(case, seed, x, past)
    if kind == "prefill_f32":
        return dict(rows=x[:-1], next=x[-1])
    if kind == "decode_f32":
        return [dict(hidden=h) for h in x]
    head, final_norm = head.double(), final_norm.double()
    if kind == "decode":
        return [dict(hidden=h, logits=head @ _rms(h, final_norm)) for h in x]
    if kind == "prefill":
        return dict(hidden=x[-2], logits=head @ _rms(x[-2], final_norm), next=x[-1])
    return dict(ids=None, logits=head @ _rms(x[-1], final_norm))
