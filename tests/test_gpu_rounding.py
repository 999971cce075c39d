"""Rounding errors of sums against float64: their size for the order in which
each kernel adds, and that they are not one-sided.

A sum of n terms that is formed in chains errs, relative to the sum's own size
and over random terms, by U sqrt(A): U = 0.43 x 2^-24 is the root mean square
of one fp32 rounding (uniform within half an ulp, mantissas spread evenly over
their logarithm), and A the mean over all roundings of the variance that the
partial sum rounded has, as a share of the whole's. A chain of c terms of n
adds (c + 1) / 2 to A, each level of a tree 1, a rounded factor 1. The chains
stated are those of a lane that adds one weight at a time, or of the matrix
kernel with k over eight waves: what these calls were always summed as."""
import numpy as np
import pytest

from nutllm_amd import workloads as W
from test_gpu_matvec_ragged import dequantised

pytestmark = pytest.mark.gpu

U = 0.43 * 2.0 ** -24
BOTH = pytest.mark.parametrize("qtype", [0, 1], ids=["int8", "int4"])


def rel(got, want):
    return np.linalg.norm(got - want) / np.linalg.norm(want)


def lane_sum(n):
    """One weight at a time over 64 lanes, then six levels of a tree."""
    return (-(-n // 64) + 1) / 2 + 6


def rms(x):
    return x / np.sqrt((x * x).mean(-1, keepdims=True) + 1e-5)


def value_rows(gpu, cfg, qtype, block, ids, path=0):
    """The V rows that a one-layer model's prompt (one token: decode step)
    leaves in the cache, and their float64 values."""
    rng = np.random.default_rng(cfg.dim + block)
    dim, ffn, kvd = cfg.dim, cfg.ffn_dim, cfg.kv_heads * cfg.head_dim
    shapes = dict(query=(dim, dim), key=(kvd, dim), value=(kvd, dim), output=(dim, dim),
                  gate=(ffn, dim), up=(ffn, dim), down=(dim, ffn))
    emb = rng.standard_normal((cfg.vocab_size, dim)).astype(np.float32)
    norm = (1 + 0.1 * rng.standard_normal(dim)).astype(np.float32)
    mats = {}
    for name, (r, c) in shapes.items():
        w = (rng.standard_normal((r, c)) * c ** -0.5).astype(np.float32)
        mats[name] = (*gpu.quantize(w, qtype, block), r, c, block)
    m, cache = gpu.DeviceModel(cfg, qtype), gpu.KVCache(cfg)
    try:
        m.set_globals(emb, np.ones(dim, np.float32), emb)
        m.set_layer(0, mats, norm, norm)
        m.set_path(path)
        if len(ids) == 1:
            m.decode(cache, int(ids[0]))
        else:
            m.prefill(cache, np.asarray(ids, np.int32))
        _, v = cache.read_positions(0, len(ids))
        got = np.asarray(v[0], np.float64).transpose(1, 0, 2).reshape(len(ids), kvd)
    finally:
        cache.close(), m.close()
    data, scales = mats["value"][:2]
    w = dequantised(data, scales, kvd, dim, qtype, block)
    return got, rms(emb[ids].astype(np.float64)) * norm @ w.T


def one_layer(gpu, heads, kv_heads, head_dim, ffn, max_seq=160):
    return gpu.Config(layers=1, heads=heads, dim=heads * head_dim, head_dim=head_dim, ffn_dim=ffn,
                      vocab_size=300, kv_heads=kv_heads, max_seq=max_seq, eos_token=1)


@BOTH
@pytest.mark.parametrize("cols,block", [(64, 64), (256, 64), (512, 128)])
def test_wide_blocks_err_as_a_lane_sum(gpu, qtype, cols, block):
    """Blocks of 64 and wider on the row kernels: 8 % over the lane sum's error
    (4,096 outputs settle it to 1 %)."""
    rng = np.random.default_rng(cols)
    rows = 4096
    data, scales = gpu.quantize(rng.standard_normal((rows, cols)).astype(np.float32), qtype, block)
    x = rng.standard_normal(cols).astype(np.float32)
    y = gpu.matvec_quantized(data, scales, rows, cols, qtype, x, block)
    want = dequantised(data, scales, rows, cols, qtype, block) @ x.astype(np.float64)
    assert rel(y, want) <= 1.08 * U * np.sqrt(lane_sum(cols))


@BOTH
@pytest.mark.parametrize("block", [64, 128])
def test_wide_blocks_err_as_a_lane_sum_in_general_steps(gpu, qtype, block):
    """The general step kernels (head size 32) at blocks of 64 and wider: x is
    scaled and weighted before (two roundings); 256 outputs settle the error
    to 5 %, the bound is 25 % over it."""
    got, want = value_rows(gpu, one_layer(gpu, 8, 8, 32, 512), qtype, block, [7])
    assert rel(got, want) <= 1.25 * U * np.sqrt(lane_sum(256) + 2)


@BOTH
@pytest.mark.parametrize("cols,block", [(33, 16), (100, 32), (255, 32), (500, 64)])
def test_straddled_blocks_err_as_a_lane_sum(gpu, qtype, cols, block):
    rng = np.random.default_rng(cols)
    rows = 4096
    data, scales = gpu.quantize(rng.standard_normal((rows, cols)).astype(np.float32), qtype, block)
    x = rng.standard_normal(cols).astype(np.float32)
    y = gpu.matvec_quantized(data, scales, rows, cols, qtype, x, block)
    want = dequantised(data, scales, rows, cols, qtype, block) @ x.astype(np.float64)
    assert rel(y, want) <= 1.08 * U * np.sqrt(lane_sum(cols))


@pytest.mark.parametrize("mkn", [(960, 2048, 960), (960, 256, 960), (960, 128, 960),
                                 (32, 128, 32)])
def test_matmul_errs_as_eight_waves(gpu, mkn):
    """k in eight chains, three levels of a tree, where 64 x 64 tiles leave
    CUs idle."""
    m, k, n = mkn
    rng = np.random.default_rng(k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((k, n)).astype(np.float32)
    want = a.astype(np.float64) @ b.astype(np.float64)
    assert rel(gpu.matmul_f32(a, b), want) <= 1.1 * U * np.sqrt((k / 8 + 1) / 2 + 3)


@pytest.mark.parametrize("heads,kv_heads,head_dim", [(8, 2, 16), (8, 4, 32), (4, 2, 64), (2, 2, 128)])
def test_attention_error_does_not_grow_with_the_keys(gpu, heads, kv_heads, head_dim):
    """A layer whose hidden state is its attention's result (V and Wo select
    dimensions, V large beside the embeddings), 1,200 keys. Scores in two
    chains; P V in chains of 16 keys, a tree over a block's (64 keys, 32 at
    head size 128), the blocks one after the other; 1.7 times that for the
    exponentials and the rescaling. One chain over all keys, 600 in A, would
    be three times the bound."""
    rng = np.random.default_rng(head_dim)
    tokens, dim, kvd = 1200, heads * head_dim, kv_heads * head_dim
    cfg = gpu.Config(layers=1, heads=heads, dim=dim, head_dim=head_dim, ffn_dim=16, vocab_size=2000,
                     kv_heads=kv_heads, max_seq=tokens, eos_token=1)
    emb = (0.1 * rng.standard_normal((2000, dim))).astype(np.float32)
    w = {name: (rng.standard_normal((dim, n)) * dim ** -0.5).astype(np.float32)
         for name, n in (("query", dim), ("key", kvd))}
    w["value"] = (1024.0 * np.eye(dim, kvd)).astype(np.float32)
    w["output"] = np.eye(dim, dtype=np.float32)
    w.update(gate=np.zeros((dim, 16), np.float32), up=np.zeros((dim, 16), np.float32),
             down=np.zeros((16, dim), np.float32))
    ones = np.ones(dim, np.float32)
    m, cache = gpu.DeviceFModel(cfg, tied=True), gpu.KVCache(cfg)
    try:
        m.set_globals(emb, ones)
        m.set_layer(0, w, ones, ones)
        ids = rng.integers(2, 2000, tokens).astype(np.int32)
        rows = m.prefill(cache, ids)[-64:].astype(np.float64)
        k, v = (np.asarray(t[0], np.float64) for t in cache.read_positions(0, tokens))
    finally:
        cache.close(), m.close()
    x = emb[ids].astype(np.float64)
    q = (rms(x) @ w["query"].astype(np.float64)).reshape(tokens, heads, head_dim)
    angle = (np.arange(tokens)[:, None] * 10000.0 ** (-2.0 * np.arange(head_dim // 2) / head_dim))
    cos, sin = np.cos(angle)[:, None], np.sin(angle)[:, None]
    q = np.stack((q[..., 0::2] * cos - q[..., 1::2] * sin,
                  q[..., 0::2] * sin + q[..., 1::2] * cos), -1).reshape(q.shape)[-64:]
    want = x[-64:].copy()
    for h in range(heads):
        s = q[:, h] @ k[h * kv_heads // heads].T / np.sqrt(head_dim)
        s[np.arange(tokens)[None] > np.arange(tokens - 64, tokens)[:, None]] = -np.inf
        p = np.exp(s - s.max(-1, keepdims=True))
        want[:, h * head_dim:(h + 1) * head_dim] += (p / p.sum(-1, keepdims=True)
                                                    @ v[h * kv_heads // heads])
    block = 32 if head_dim == 128 else 64
    terms = (head_dim / 2 + 1) / 2 + 1 + 17 / 2 + 2 + tokens / block / 2
    assert rel(rows, want) <= 1.7 * U * np.sqrt(terms)


@BOTH
@pytest.mark.parametrize("tokens", [16, 64])
def test_row_tiles_round_to_both_sides(gpu, qtype, tokens):
    """The errors of a prompt's V rows on the row tiles have no common sign (an
    MFMA that adds large products to a small C rounds that down, 0.4 of the
    error on average): 0.1 is several times the spread of the mean over 1,024
    or more outputs of about one rounding each."""
    got, want = value_rows(gpu, one_layer(gpu, 16, 4, 64, 1024), qtype, 32,
                           np.arange(3, 3 + tokens))
    error = got - want
    assert abs(error.mean()) <= 0.1 * np.sqrt((error * error).mean())


@BOTH
@pytest.mark.parametrize("tokens", [2, 20, 70])
def test_dense_prompts_err_as_short_chains(gpu, qtype, tokens):
    """Prompts whose weights are written out as fp32 (head size 32, blocks of
    48): a chunk of 32 k in four chains and two levels, three over the waves,
    and the row's two factors; 512 outputs and more settle it to 4 %, the bound
    is 15 % over it. One chain per chunk and the waves one after the other,
    23 in A, would be 20 % over the bound."""
    got, want = value_rows(gpu, one_layer(gpu, 8, 8, 32, 512), qtype, 48,
                           np.arange(3, 3 + tokens))
    assert rel(got, want) <= 1.15 * U * np.sqrt((8 + 1) / 2 + 2 + 3 + 2)
