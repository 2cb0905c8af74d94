"""A mixture's experts in a prompt block of up to 128 tokens, all of a layer in one launch (prefill.hip): experts of one token tile, of several and of full blocks (two experts, both of every token), experts
nobody chose, one expert a token, k in ranges of one block, of several (gate | up of eight experts 8192 wide and of two 10240 wide, down in ranges of two and four) and with a last range that is shorter, in every format,
against the exact token-by-token path.

Tolerance as in test_gpu_prefill.py: operands of the blocks are rounded to f16."""
import block_rows
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mix,kw,sizes", [
    ("Q4_K_M", dict(num_experts=2, num_experts_per_token=2), (3, 97, 128)),
    ("Q8_0", dict(num_experts=2, num_experts_per_token=2, expert_intermediate_size=1024), (128,)),
    ("Q5_K_M", dict(num_experts=8, num_experts_per_token=2, expert_intermediate_size=2048), (2, 16, 63, 128)),
    ("Q6_K", dict(num_experts=1, num_experts_per_token=1), (128,)),
    ("Q4_0", dict(num_experts=5, num_experts_per_token=1, expert_intermediate_size=1792), (40, 113)),
])
def test_block_of_a_mixture_matches_token_by_token(pkg, mix, kw, sizes):
    cfg = pkg.make_config("test-moe", max_seq_len=160, **kw)
    model = pkg.SynthModel(cfg, mix=mix)
    exact = pkg.HipGpuInference.from_model(model, 160, flags=pkg.hip_backend.FLAG_EXACT_PREFILL)
    block = pkg.HipGpuInference.from_model(model, 160)
    assert block.prefill_is_batched()
    for m in sizes:
        prompt = [(11 * i + 5) % cfg.vocab_size for i in range(m)]
        out = []
        for eng in (exact, block):
            eng.reset()
            eng.forward_batch(prompt)
            out.append(eng.forward(9))
        want, got = out
        assert np.abs(got - want).max() <= 1e-2 * np.abs(want).max() + 1e-2, (m, np.abs(got - want).max())
    exact.close()
    block.close()


@pytest.mark.parametrize("mix,experts,top_k,hidden,ff,tokens", [
    ("Q4_K_M", 2, 2, 2048, 10240, (33, 64, 97, 128)),     # gate | up in ranges of three, three and two blocks, full experts
    ("Q8_0", 2, 2, 2048, 10240, (65, 128)),
    ("Q5_K_M", 8, 2, 2048, 8192, (20, 100, 128)),         # in one of eight blocks; some experts of two token tiles, some of more
    ("Q6_K", 8, 2, 2048, 8192, (128,)),
    ("Q4_0", 8, 2, 2048, 8192, (128,)),
    ("Q5_K_M", 8, 2, 512, 2048, (16, 128)),               # one block a range
])
def test_rows_behind_a_block(pkg, mix, experts, top_k, hidden, ff, tokens):
    kw = dict(num_experts=experts, num_experts_per_token=top_k, hidden_size=hidden, expert_intermediate_size=ff, num_layers=2)
    block_rows.check(pkg, pkg.SynthModel(pkg.make_config("test-moe", max_seq_len=160, **kw), mix=mix), tokens)
