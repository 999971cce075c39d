"""Calls on a device without memory for their workspace: what needs one fails
with DeviceError and leaves the model as usable as before, and what has a way
without one goes that way."""
import numpy as np
import pytest

from nutllm_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture
def scarce(gpu):
    yield gpu.fail_allocations
    gpu.fail_allocations(0, 0)


# the step kernels' chunk, the row tiles, the batch (step_gqa2), and a greedy
# loop on the graph
@pytest.mark.parametrize("tokens,generated", [(3, 0), (20, 0), (150, 0), (3, 4)])
def test_failed_workspace_leaves_the_model_usable(gpu, scarce, tokens, generated):
    """Every allocation of a model's first call fails once, in turn."""
    host = W.build("step_gqa2", 1, 7, max_seq=200)
    ids = gpu.synth_tokens(9, host.config.vocab_size, tokens).astype(np.int32)
    cache = gpu.KVCache(host.config)

    def call(model):
        return model.generate(ids, generated)[0] if generated else model.prefill(cache, ids)

    model = host.to_device()
    want = call(model)
    model.close()
    failed = 0
    for skip in range(40):
        model = host.to_device()
        try:
            scarce(skip, 1)
            call(model)
            break
        except gpu.DeviceError as error:
            assert "memory" in str(error)
            failed += 1
            scarce(0, 0)
            assert np.array_equal(call(model), want)
        finally:
            scarce(0, 0)
            model.close()
    else:
        pytest.fail("the call never ran out of allocations")
    assert failed >= 2
    cache.close()


@pytest.mark.parametrize("count", [1, 3, 100])
@pytest.mark.parametrize("qtype", [0, 1], ids=["int8", "int4"])
def test_dense_prompt_without_memory_runs_token_by_token(gpu, scarce, qtype, count):
    host = W.build("tiny", qtype, 7)
    ids = gpu.synth_tokens(9, host.config.vocab_size, 20).astype(np.int32)
    model, cache, steps = host.to_device(), gpu.KVCache(host.config), gpu.KVCache(host.config)
    try:
        model.set_path(1)
        want = model.prefill(steps, ids)
        model.set_path(0)
        scarce(5 - min(count, 5), count)
        assert np.array_equal(model.prefill(cache, ids), want)
        scarce(0, 0)
        for a, b in zip(cache.read_positions(0, 20), steps.read_positions(0, 20)):
            assert np.array_equal(a, b)
        assert np.array_equal(model.decode(cache, 3), model.decode(steps, 3))
        again = model.prefill(cache, ids)  # with memory again: the dense form
        assert np.linalg.norm(again - want) <= 5e-6 * np.linalg.norm(want)
    finally:
        model.close(), cache.close(), steps.close()


@pytest.mark.parametrize("count", [1, 3, 100])
@pytest.mark.parametrize("head_dim", [64, 48])
def test_fp32_prompt_without_memory_runs_token_by_token(gpu, scarce, head_dim, count):
    rng = np.random.default_rng(head_dim)
    dim, ffn = 2 * head_dim, 100
    cfg = gpu.Config(layers=2, heads=2, dim=dim, head_dim=head_dim, ffn_dim=ffn, vocab_size=50,
                     kv_heads=1, max_seq=64, eos_token=1)
    dims = dict(query=(dim, dim), key=(dim, head_dim), value=(dim, head_dim), output=(dim, dim),
                gate=(dim, ffn), up=(dim, ffn), down=(ffn, dim))
    model, cache, steps = gpu.DeviceFModel(cfg, tied=True), gpu.KVCache(cfg), gpu.KVCache(cfg)
    ones = np.ones(dim, np.float32)
    try:
        model.set_globals(rng.standard_normal((50, dim)).astype(np.float32), ones)
        for layer in range(2):
            model.set_layer(layer, {k: (rng.standard_normal(s) * s[0] ** -0.5).astype(np.float32)
                                    for k, s in dims.items()}, ones, ones)
        ids = rng.integers(2, 50, 20).astype(np.int32)
        want = np.stack([model.decode(steps, int(t)) for t in ids])
        scarce(5 - min(count, 5), count)
        assert np.array_equal(model.prefill(cache, ids), want)
        scarce(0, 0)
        assert np.array_equal(model.decode(cache, 3), model.decode(steps, 3))
        again = model.prefill(cache, ids)  # with memory again: as a batch
        assert np.linalg.norm(again - want) <= 5e-6 * np.linalg.norm(want)
    finally:
        model.close(), cache.close(), steps.close()
