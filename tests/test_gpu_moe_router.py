"""The decode router (misc.hip, moe_router_kernel) through whole tokens against the CPU oracle, at the ends of its ranges: as many experts as a wave has lanes, fewer than waves, more columns than a pass of a
wave holds (4096) and than the one-round-trip form takes (8192).  Tolerance of a decode step: 2e-3 of the largest logit + 2e-3 (a wrong expert moves logits by far more)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,experts,top_k", [(512, 64, 8), (256, 3, 1), (768, 9, 4), (4352, 10, 2), (8448, 4, 2)])
def test_router_picks_the_oracles_experts(pkg, orc, hidden, experts, top_k):
    cfg = pkg.make_config("test-moe", max_seq_len=16, hidden_size=hidden, num_layers=2, vocab_size=256, num_experts=experts, num_experts_per_token=top_k, expert_intermediate_size=256)
    model = pkg.SynthModel(cfg, mix="Q4_0")
    ref = orc.Model(cfg.as_dict())
    for nm, t, ne, data in model.tensors(keep=True):
        ref.add_tensor(nm, t, ne, data)
    ref.finalize()
    eng = pkg.HipGpuInference.from_model(model, 16)
    for tok in (3, 200, 77, 5):
        got, want = eng.forward(tok), ref.forward([tok])
        assert np.abs(got - want).max() <= 2e-3 * np.abs(want).max() + 2e-3
    eng.close()
