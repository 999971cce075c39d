"""The fp32 path's prompt batches and decode steps against a float64 numpy
transformer, at the edges of their tiles: one row, one less and one more than
a 16-row attention tile and a 64-key block, head sizes with an attention kernel
of their own and one without, widths that no 32-wide k chunk divides, and one
layer of real widths at the lengths that take each GEMM tile in each of the
projections, k whole and in two, three and four runs (tile_choice.py says which
a case takes, test_cpu_tiles.py that they are all there).

The bound on the relative error (2-norm) is 5e-6 per call: an fp32 chain of k
terms errs by about sqrt(k) 2^-24 / 4 relative to its rms, k <= 300 here, or at
the real widths, whose waves share k, k <= 1,500, over two layers or one of five
products each (about 1e-6), with a factor of five to spare."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# heads, kv_heads, head_dim, ffn, vocab
SHAPES = {
    "hd16": (4, 2, 16, 172, 97),
    "hd32": (3, 3, 32, 100, 50),
    "hd64": (4, 1, 64, 300, 64),
    "hd128": (2, 2, 128, 257, 40),
    "hd48": (2, 1, 48, 130, 33),
    "long": (2, 1, 64, 4131, 30),  # W2's k in runs, the last with a tail
}
# one layer each: the shape and the prompt lengths that are tested with it
WIDE = {
    "w2048": ((32, 4, 64, 5632, 64), (40, 301)),
    "w2560": ((20, 2, 128, 4100, 64), (16, 301)),
    "w4096": ((32, 16, 128, 4200, 64), (1, 16, 40, 80, 180, 200)),
    "w4096n": ((32, 1, 128, 1100, 64), (16,)),
}


def rms(x, w):
    return x / np.sqrt((x * x).mean(-1, keepdims=True) + 1e-5) * w


def rope(x, first):
    t, _, hd = x.shape
    a = (np.arange(first, first + t)[:, None] * 10000.0 ** (-2.0 * np.arange(hd // 2) / hd))[:, None]
    out = np.empty_like(x)
    out[..., 0::2] = x[..., 0::2] * np.cos(a) - x[..., 1::2] * np.sin(a)
    out[..., 1::2] = x[..., 0::2] * np.sin(a) + x[..., 1::2] * np.cos(a)
    return out


class Exact:
    def __init__(self, cfg, emb, layers):
        self.c, self.emb, self.layers = cfg, emb.astype(np.float64), layers
        self.k = [None] * cfg.layers
        self.v = [None] * cfg.layers

    def run(self, ids, first):
        c = self.c
        x = self.emb[ids]
        t = len(ids)
        for i, (w, an, fn) in enumerate(self.layers):
            h = rms(x, an)
            q = rope((h @ w["query"]).reshape(t, c.heads, c.head_dim), first)
            k = rope((h @ w["key"]).reshape(t, c.kv_heads, c.head_dim), first)
            v = (h @ w["value"]).reshape(t, c.kv_heads, c.head_dim)
            self.k[i] = k if first == 0 else np.concatenate((self.k[i], k))
            self.v[i] = v if first == 0 else np.concatenate((self.v[i], v))
            rep = c.heads // c.kv_heads
            s = np.einsum("thd,phd->htp", q, np.repeat(self.k[i], rep, 1)) / np.sqrt(c.head_dim)
            n = self.k[i].shape[0]
            s[:, np.arange(n)[None] > np.arange(first, first + t)[:, None]] = -np.inf
            p = np.exp(s - s.max(-1, keepdims=True))
            p /= p.sum(-1, keepdims=True)
            ctx = np.einsum("htp,phd->thd", p, np.repeat(self.v[i], rep, 1)).reshape(t, -1)
            x = x + ctx @ w["output"]
            h = rms(x, fn)
            g = h @ w["gate"]
            x = x + (g / (1 + np.exp(-g)) * (h @ w["up"])) @ w["down"]
        return x


def build(gpu, shape, rng, vocab_fill=None, count=2):
    heads, kvh, hd, ffn, vocab = SHAPES[shape] if shape in SHAPES else WIDE[shape][0]
    dim = heads * hd
    cfg = gpu.Config(layers=count, heads=heads, dim=dim, head_dim=hd, ffn_dim=ffn, vocab_size=vocab,
                     kv_heads=kvh, max_seq=320, eos_token=1)
    emb = rng.standard_normal((vocab, dim)).astype(np.float32)
    if vocab_fill is not None:
        emb[vocab_fill[0]] = vocab_fill[1]
    dims = dict(query=(dim, dim), key=(dim, kvh * hd), value=(dim, kvh * hd), output=(dim, dim),
                gate=(dim, ffn), up=(dim, ffn), down=(ffn, dim))
    m = gpu.DeviceFModel(cfg, tied=True)
    m.set_globals(emb, np.ones(dim, np.float32))
    layers = []
    for i in range(count):
        w = {k: (rng.standard_normal(s, np.float32) * s[0] ** -0.5).astype(np.float32)
             for k, s in dims.items()}
        an, fn = ((1 + 0.1 * rng.standard_normal(dim)).astype(np.float32) for _ in range(2))
        m.set_layer(i, w, an, fn)
        layers.append(({k: v.astype(np.float64) for k, v in w.items()}, an.astype(np.float64),
                       fn.astype(np.float64)))
    return cfg, m, Exact(cfg, emb, layers)


@pytest.mark.parametrize("tokens", [1, 2, 15, 16, 17, 64, 65, 300])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_batch_and_steps_match_float64(gpu, shape, tokens):
    rng = np.random.default_rng(tokens)
    cfg, m, exact = build(gpu, shape, rng)
    cache = gpu.KVCache(cfg)
    try:
        ids = rng.integers(2, cfg.vocab_size, tokens).astype(np.int32)
        rows, want = m.prefill(cache, ids), exact.run(ids, 0)
        assert np.linalg.norm(rows - want) <= 5e-6 * np.linalg.norm(want)
        for step in range(2):
            token = int(rng.integers(2, cfg.vocab_size))
            got, want = m.decode(cache, token), exact.run([token], tokens + step)[0]
            assert np.linalg.norm(got - want) <= 5e-6 * np.linalg.norm(want)
        k, v = cache.read_positions(0, tokens + 2)
        for i in range(2):
            want = exact.v[i].transpose(1, 0, 2)
            assert np.linalg.norm(v[i] - want) <= 5e-6 * np.linalg.norm(want)
    finally:
        cache.close()
        m.close()


@pytest.mark.parametrize("shape", list(WIDE))
def test_real_widths_match_float64(gpu, shape):
    rng = np.random.default_rng(17)
    cfg, m, exact = build(gpu, shape, rng, count=1)
    cache = gpu.KVCache(cfg)
    try:
        for tokens in WIDE[shape][1]:
            ids = rng.integers(2, cfg.vocab_size, tokens).astype(np.int32)
            rows, want = m.prefill(cache, ids), exact.run(ids, 0)
            print(shape, tokens, flush=True)
            # row by row: a row tile or a column tile that went wrong shows
            error = np.linalg.norm(rows - want, axis=1)
            assert np.all(error <= 5e-6 * np.linalg.norm(want, axis=1))
            assert np.all(np.abs(rows - want) <= 5e-5 * np.sqrt((want * want).mean()))
            k, v = cache.read_positions(0, tokens)
            for got, ref in ((k[0], exact.k[0]), (v[0], exact.v[0])):
                assert np.linalg.norm(got - ref.transpose(1, 0, 2)) <= 5e-6 * np.linalg.norm(ref)
    finally:
        cache.close()
        m.close()


@pytest.mark.parametrize("shape", ["hd16", "hd64", "hd128"])
def test_non_finite_token_leaves_earlier_rows(gpu, shape):
    """A token whose embedding is not finite spoils its own row and the later
    ones, none before it."""
    rng = np.random.default_rng(3)
    cfg, m, exact = build(gpu, shape, rng, vocab_fill=(7, np.nan))
    cache = gpu.KVCache(cfg)
    try:
        ids = rng.integers(8, cfg.vocab_size, 40).astype(np.int32)
        ids[21] = 7
        rows = m.prefill(cache, ids)
        want = exact.run(ids[:21], 0)
        assert np.linalg.norm(rows[:21] - want) <= 5e-6 * np.linalg.norm(want)
        assert not np.any(np.isfinite(rows[21:]))
    finally:
        cache.close()
        m.close()


@pytest.mark.parametrize("head_dim", [48, 64, 128])
@pytest.mark.parametrize("hidden", [31, 32, 200])
def test_keys_at_minus_infinity_have_no_weight(gpu, head_dim, hidden):
    """A decode step over keys whose scores overflow to minus infinity (whole
    runs of the split attention among them) and five ordinary ones after them:
    the ordinary ones alone count, as in one softmax over all."""
    rng = np.random.default_rng(hidden)
    SHAPES["inf"] = (2, 2, head_dim, 100, 50)
    cfg, m, exact = build(gpu, "inf", rng, count=1)
    cache = gpu.KVCache(cfg)
    try:
        token = 7
        w, an, _ = exact.layers[0]
        q = rope((rms(exact.emb[[token]], an) @ w["query"]).reshape(1, 2, head_dim), hidden + 5)[0]
        k = rng.standard_normal((hidden + 5, 2, head_dim)).astype(np.float32)
        v = rng.standard_normal((hidden + 5, 2, head_dim)).astype(np.float32)
        k[:hidden] = -3e38 * np.sign(q)
        cache.write_positions(0, k.transpose(1, 0, 2)[None], v.transpose(1, 0, 2)[None])
        exact.k[0], exact.v[0] = k.astype(np.float64), v.astype(np.float64)
        cache.set_length(hidden + 5)
        got, want = m.decode(cache, token), exact.run([token], hidden + 5)[0]
        assert np.linalg.norm(got - want) <= 5e-6 * np.linalg.norm(want)
    finally:
        del SHAPES["inf"]
        cache.close()
        m.close()
