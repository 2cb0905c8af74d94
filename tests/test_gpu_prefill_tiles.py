"""Token tiles of 96 to 256 in steps of 32 (prefill_wide.hip, pw_body): a prompt's last tile at both edges of each, with formats of three activation buffers and of two; a mixture whose experts get some 40 to 200 rows.

Against the exact engine (f32 throughout, token by token), with the tolerance of the other long prompts: operands are rounded to f16 (2^-12 each), and a layer's rounding is carried on by the next ones: 1e-2 of the largest
logit, of which 1e-3 to 3e-3 are measured.  (That bound is for tokens whose experts both engines choose alike: behind 800 of these tokens a router's close call falls to the other side after that rounding, 1.3e-2 with
tiles of 256, 192 and 128 alone, too, and with the same bits.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,mix,sizes", [
    ("test-dense", "Q4_K_M", (257, 289, 320, 352, 353, 416, 417, 480, 481)), ("test-dense", "Q8_0", (288, 352, 385, 416, 449, 480)), ("test-dense", "Q6_K", (340, 400, 470)),
    ("test-dense-d128", "Q5_K_M", (345, 411, 476)), ("test-dense", "Q4_0", (351, 415, 479)), ("test-moe", "Q5_K_M", (170, 300, 450, 620)),
])
def test_last_tiles_match_the_exact_engine(pkg, name, mix, sizes):
    cap = max(sizes) + 8
    cfg = pkg.make_config(name, max_seq_len=cap)
    model = pkg.SynthModel(cfg, mix=mix)
    exact, wide = pkg.HipGpuInference.from_model(model, cap, flags=pkg.hip_backend.FLAG_EXACT_PREFILL), pkg.HipGpuInference.from_model(model, cap)
    prompt = [(7 * i + 3) % cfg.vocab_size for i in range(max(sizes))]
    for n in sizes:
        for eng in (exact, wide):
            eng.reset()
            eng.forward_batch(prompt[:n])
        for t in (5, 77):
            want, got = exact.forward(t), wide.forward(t)
            assert np.abs(got - want).max() <= 1e-2 * float(np.abs(want).max()) + 1e-2, (n, t)
    exact.close()
    wide.close()
