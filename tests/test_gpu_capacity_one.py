"""Contexts that hold a single position: what is launched ahead of the first token, when the context and its slots are made, stays at position 0, and the one token's logits are the larger context's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model,mix", [("test-dense-d128", "Q4_K_M"), ("test-moe", "Q5_K_M")])
def test_one_token(pkg, model, mix):
    m = pkg.SynthModel(pkg.make_config(model, max_seq_len=40), mix=mix)
    one, more = pkg.HipGpuInference.from_model(m, 1), pkg.HipGpuInference.from_model(m, 40)
    for token in (7, 3):
        one.reset()
        more.reset()
        assert np.array_equal(one.forward(token).view(np.uint32), more.forward(token).view(np.uint32))
        with pytest.raises(pkg.hip_backend.BackendError):
            one.forward(token)
    one.close()
    more.close()


@pytest.mark.parametrize("slots", [1, 3])
def test_one_token_a_slot(pkg, slots):
    cfg = pkg.make_config("test-dense-d128", max_seq_len=1, num_layers=2)
    eng = pkg.HipGpuInference.from_model(pkg.SynthModel(cfg, mix="Q4_K_M"), 1)
    eng.batch_create(slots)
    got, _ = eng.forward_multi(list(range(slots)), [7 + s for s in range(slots)])
    for s in range(slots):
        eng.reset()
        assert np.array_equal(got[s].view(np.uint32), eng.forward(7 + s).view(np.uint32))
    with pytest.raises(pkg.hip_backend.BackendError):
        eng.forward_multi([0], [1])
    eng.close()
