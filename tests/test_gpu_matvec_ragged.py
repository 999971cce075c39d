"""The quantised matvec where blocks straddle rows and at block sizes of 64 and
128, at the edges of its runs of 16 weights, and a decode step at block 64.

Against a float64 product of the dequantised weights; every output's error is
bounded by (terms a lane adds + 6 reduction steps + 2) 2^-23 sum |w x|, doubled
for the offset-binary form of the whole-block kernels, whose codes run to twice
their size."""
import numpy as np
import pytest

from nutllm_amd import workloads as W

pytestmark = pytest.mark.gpu


def dequantised(data, scales, rows, cols, qtype, block):
    n = rows * cols
    raw = np.asarray(data).view(np.uint8)
    if qtype == 1:
        q = np.empty(raw.size * 2, np.int8)
        q[0::2], q[1::2] = raw & 15, raw >> 4
        q = np.where(q >= 8, q - 16, q)[:n]
    else:
        q = raw.view(np.int8)[:n]
    s = np.asarray(scales).view(np.float16).astype(np.float64)
    return (q.astype(np.float64) * np.repeat(s, block)[:n]).reshape(rows, cols)


@pytest.mark.parametrize("qtype", [0, 1], ids=["int8", "int4"])
@pytest.mark.parametrize("rows,cols,block", [
    (1, 16, 32), (3, 15, 32), (16, 17, 16), (17, 1039, 32), (33, 1025, 64), (31, 3001, 32),
    (5, 1056, 64), (40, 2048, 64), (2050, 1024, 128), (9, 96, 32), (6, 672, 512), (7, 333, 24),
    (3, 14001, 32),
])
def test_matvec_any_block_layout(gpu, qtype, rows, cols, block):
    rng = np.random.default_rng(rows * 31 + cols)
    w = rng.standard_normal((rows, cols)).astype(np.float32)
    x = rng.standard_normal(cols).astype(np.float32)
    data, scales = gpu.quantize(w, qtype, block)
    y = gpu.matvec_quantized(data, scales, rows, cols, qtype, x, block)
    d = dequantised(data, scales, rows, cols, qtype, block)
    bound = 2 * (cols / 64 + 24) * 2.0 ** -23 * (np.abs(d) @ np.abs(x).astype(np.float64))
    # the offset-binary form adds bias * s * |x| to what is summed
    step = np.abs(d).max() / (7 if qtype else 127)
    bound += 24 * 2.0 ** -23 * step * (8 if qtype else 128) * np.abs(x).sum()
    assert np.all(np.abs(y - d @ x.astype(np.float64)) <= bound)


@pytest.mark.parametrize("qtype", [0, 1], ids=["int8", "int4"])
@pytest.mark.parametrize("block", [64, 128, 48])
def test_decode_step_other_blocks(gpu, qtype, block):
    """A model whose blocks are 64 or 128 wide runs the step kernels, one of
    48 the general ones: both within the parity bar of the same weights
    as an oracle model, over a prompt and the steps after it."""
    cfg = W.make_config("step_gqa2", max_seq=96)
    rng = np.random.default_rng(block)
    dim, ffn, kvd = cfg.dim, cfg.ffn_dim, cfg.kv_heads * cfg.head_dim
    shapes = dict(query=(dim, dim), key=(kvd, dim), value=(kvd, dim), output=(dim, dim),
                  gate=(ffn, dim), up=(ffn, dim), down=(dim, ffn))
    emb = rng.standard_normal((cfg.vocab_size, dim)).astype(np.float32)
    ones = np.ones(dim, np.float32)
    a, b = gpu.DeviceModel(cfg, qtype), gpu.DeviceFModel(cfg, tied=True)
    a.set_globals(emb, ones, emb)
    b.set_globals(emb, ones)
    for i in range(cfg.layers):
        mats, dense = {}, {}
        for name, (r, c) in shapes.items():
            w = (rng.standard_normal((r, c)) * c ** -0.5).astype(np.float32)
            data, scales = gpu.quantize(w, qtype, block)
            mats[name] = (data, scales, r, c, block)
            # the products q s are exact in fp32: 8 and 11 bits
            dense[name] = np.ascontiguousarray(
                dequantised(data, scales, r, c, qtype, block).T.astype(np.float32))
        a.set_layer(i, mats, ones, ones)
        b.set_layer(i, dense, ones, ones)
    ca, cb = gpu.KVCache(cfg), gpu.KVCache(cfg)
    try:
        ids = rng.integers(2, cfg.vocab_size, 37).astype(np.int32)
        got, want = a.prefill(ca, ids), b.prefill(cb, ids)[-1]
        assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
        for _ in range(2):
            token = int(rng.integers(2, cfg.vocab_size))
            got, want = a.decode(ca, token), b.decode(cb, token)
            assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
    finally:
        ca.close(), cb.close(), a.close(), b.close()


def test_matvec_rows_past_one_grid(gpu):
    """More rows than a grid of a workgroup per 16 rows covers (2^32 threads):
    codes times scales of one, which are exact."""
    rows = 140_000_000
    data = (np.arange(rows) % 251 - 125).astype(np.int8)
    scales = np.full((rows + 31) // 32, 0x3c00, np.uint16)
    y = gpu.matvec_quantized(data.view(np.uint8), scales, rows, 1, 0,
                             np.full(1, 0.5, np.float32))
    assert np.array_equal(y, np.float32(0.5) * data)
