"""gate | up of a prompt block as one product without partial sums (prefill.hip) against the exact token-by-token path: token counts around the tiles of 32 and the largest of each kernel; up to 32 tokens over k in
multiples of 1024, two teams of waves with half of k each (pf_pair_few_kernel: its loop takes two blocks a turn, one turn at 1024 columns, two and four at 2048 and 4096), all others with halves of every block
(pf_pair_kernel: three blocks a turn, none, one or two left over), narrow widths and some that fill the chip.

Tolerance: operands rounded to 11 bits, f32 sums, as for every product of the batched prompt path: 1e-2 of the largest logit + 1e-2."""
import block_rows
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,ff,mix,tokens", [
    (512, 768, "Q4_K_M", (2, 31, 32, 33, 64)),
    (1024, 1280, "Q5_K_M", (15, 33, 63, 65)),
    (1024, 512, "Q4_0", (32, 49, 64)),
    (2048, 768, "Q8_0", (20, 64)),
    (1024, 768, "Q6_K", (3, 61)),
    (512, 11008, "Q4_K_M", (63, 65, 96, 127, 128)),
    (1024, 11264, "Q5_K_M", (97, 128)),
    (512, 11008, "Q6_K", (66, 128)),
    (512, 11008, "Q8_0", (128,)),
])
def test_gate_up_product_matches_the_exact_path(pkg, hidden, ff, mix, tokens):
    cfg = pkg.make_config("test-dense-d128", max_seq_len=160, hidden_size=hidden, intermediate_size=ff, num_layers=3)
    model = pkg.SynthModel(cfg, mix=mix)
    exact = pkg.HipGpuInference.from_model(model, 160, flags=pkg.hip_backend.FLAG_EXACT_PREFILL)
    batched = pkg.HipGpuInference.from_model(model, 160)
    assert batched.prefill_is_batched()
    for n in tokens:
        prompt = [(11 * i + n) % cfg.vocab_size for i in range(n)]
        exact.reset()
        batched.reset()
        exact.forward_batch(prompt)
        batched.forward_batch(prompt)
        for tok in (5, 17):
            want, got = exact.forward(tok), batched.forward(tok)
            assert np.isfinite(got).all() and np.abs(got - want).max() <= 1e-2 * np.abs(want).max() + 1e-2, n
    exact.close()
    batched.close()


@pytest.mark.parametrize("hidden,ff,mix,tokens", [
    (1024, 1280, "Q4_0", (20, 32, 33)),
    (2048, 768, "Q8_0", (20, 64)),
    (2048, 5632, "Q4_K_M", (17, 31, 32, 33, 100)),
    (2048, 5632, "Q5_K_M", (17, 31, 32)),
    (2048, 5632, "Q6_K", (31,)),
    (4096, 14336, "Q8_0", (17, 32)),
    (4096, 14336, "Q4_K_M", (32, 127)),
    (4096, 11008, "Q5_K_M", (32,)),
    (1280, 2048, "Q8_0", (20, 64, 96)),       # five blocks
    (1536, 4096, "Q5_K_M", (9, 64, 128)),     # six
    (1792, 1024, "Q4_0", (32, 33, 97)),       # seven
])
def test_rows_behind_a_block(pkg, hidden, ff, mix, tokens):
    block_rows.check(pkg, pkg.SynthModel(pkg.make_config("test-dense-d128", max_seq_len=160, hidden_size=hidden, intermediate_size=ff, num_layers=2), mix=mix), tokens)
