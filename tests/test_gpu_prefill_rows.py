"""Short prompts on the row tiles, and prompts of a shape without step kernels
(tiny) on fp32 weights, against the per-token kernels.

Lengths at the edges of the tiles (16 and 32 rows) and of the range that takes
them (6 or 9 rows on at small widths; the shorter ones, and those past its end,
run on the step kernels and the batched GEMM), INT8 and INT4, head sizes 64 and
128: the last hidden state, the K/V rows of every position and the step that
follows. The bar is 5e-6 on the relative error: fp32 sums, and activations as
three bf16 limbs without a remainder, over two layers; the step kernels
themselves are within 2e-6 of 64 bits here."""
import numpy as np
import pytest

from nutllm_amd import workloads as W

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.fixture(scope="module", params=[("step_gqa2", 0), ("step_gqa4", 1), ("step_mha128", 0),
                                        ("step_mha128", 1), ("tiny", 0), ("tiny", 1)], ids=lambda p: f"{p[0]}-{p[1]}")
def model(request, gpu):
    shape, qtype = request.param
    m = W.build(shape, qtype, 31, max_seq=160, norm_seed=5)
    dev = m.to_device()
    yield m.config, dev
    dev.close()


@pytest.mark.parametrize("tokens", [2, 3, 8, 9, 15, 16, 17, 31, 32, 33, 64, 65, 127, 128,
                                    129])
def test_row_tiles_match_steps(gpu, model, tokens):
    cfg, dev = model
    ids = gpu.synth_tokens(9, cfg.vocab_size, tokens).astype(np.int32)
    rows, steps = gpu.KVCache(cfg), gpu.KVCache(cfg)
    try:
        got = dev.prefill(rows, ids)
        dev.set_path(1)
        want = dev.prefill(steps, ids)
        dev.set_path(0)
        assert rel(got, want) <= 5e-6
        for a, b in zip(rows.read_positions(0, tokens), steps.read_positions(0, tokens)):
            assert rel(a, b) <= 5e-6
        assert rel(dev.decode(rows, 3), dev.decode(steps, 3)) <= 5e-6
    finally:
        dev.set_path(0)
        rows.close(), steps.close()


# heads, kv_heads, head_dim, ffn: one layer, and the lengths tested with it, the
# last of w3072 and w4096 the shortest that the batched GEMM takes there.
# Real widths take the forms of wide outputs; layers with three query heads per
# KV head or head size 32 have no step kernels and take the tiles from 2 rows.
WIDE = {
    "w2048": ((32, 4, 64, 5632), (6, 16, 17, 40, 64)),
    "w3072": ((24, 6, 128, 1152), (5, 16, 32, 33)),
    "w4096": ((32, 8, 128, 4224), (5, 16, 17)),
    "group3": ((6, 2, 64, 640), (2, 5, 17, 128)),
    "head32": ((8, 4, 32, 384), (2, 16, 33)),
}


@pytest.mark.parametrize("qtype", [0, 1], ids=["int8", "int4"])
@pytest.mark.parametrize("shape", list(WIDE))
def test_row_tiles_match_steps_at_other_widths(gpu, qtype, shape):
    (heads, kvh, hd, ffn), lengths = WIDE[shape]
    dim, kvd = heads * hd, kvh * hd
    cfg = gpu.Config(layers=1, heads=heads, dim=dim, head_dim=hd, ffn_dim=ffn, vocab_size=400,
                     kv_heads=kvh, max_seq=160, eos_token=1)
    rng = np.random.default_rng(ffn)
    dims = dict(query=(dim, dim), key=(kvd, dim), value=(kvd, dim), output=(dim, dim),
                gate=(ffn, dim), up=(ffn, dim), down=(dim, ffn))
    mats = {}
    for name, (r, c) in dims.items():
        w = rng.standard_normal((r, c), np.float32) * np.float32(c ** -0.5)
        mats[name] = (*gpu.quantize(w, qtype), r, c)
    norms = [(1 + 0.1 * rng.standard_normal(dim)).astype(np.float32) for _ in range(2)]
    emb = rng.standard_normal((400, dim), np.float32)
    dev, rows, steps = gpu.DeviceModel(cfg, qtype), gpu.KVCache(cfg), gpu.KVCache(cfg)
    try:
        dev.set_globals(emb, norms[0], emb)
        dev.set_layer(0, mats, *norms)
        for tokens in lengths:
            ids = rng.integers(2, 400, tokens).astype(np.int32)
            got = dev.prefill(rows, ids)
            dev.set_path(1)
            want = dev.prefill(steps, ids)
            dev.set_path(0)
            assert rel(got, want) <= 5e-6
            for a, b in zip(rows.read_positions(0, tokens), steps.read_positions(0, tokens)):
                assert rel(a, b) <= 5e-6
                error = np.abs(np.asarray(a, np.float64) - b)  # no part of a tile is wrong
                assert error.max() <= 5e-5 * np.sqrt((np.asarray(b, np.float64) ** 2).mean())
            assert rel(dev.decode(rows, 3), dev.decode(steps, 3)) <= 5e-6
    finally:
        dev.set_path(0)
        dev.close(), rows.close(), steps.close()


@pytest.mark.parametrize("scale", [1e-5, 1.0, 1e8])
@pytest.mark.parametrize("qtype", [0, 1], ids=["int8", "int4"])
def test_row_tiles_take_rows_of_any_size(gpu, qtype, scale):
    """Hidden rows far below f16's smallest and far above its largest value:
    the tiles split them before they are normalised."""
    m = W.build("step_gqa4", qtype, 31, max_seq=64, norm_seed=5)
    m.embeddings = (m.embeddings * np.float32(scale)).astype(np.float32)
    dev = m.to_device()
    rows, steps = gpu.KVCache(m.config), gpu.KVCache(m.config)
    try:
        ids = gpu.synth_tokens(9, m.config.vocab_size, 20).astype(np.int32)
        got = dev.prefill(rows, ids)
        dev.set_path(1)
        want = dev.prefill(steps, ids)
        assert np.all(np.isfinite(want)) and rel(got, want) <= 5e-6
        for a, b in zip(rows.read_positions(0, 20), steps.read_positions(0, 20)):
            assert rel(a, b) <= 5e-6
    finally:
        rows.close(), steps.close(), dev.close()
