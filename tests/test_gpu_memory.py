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
