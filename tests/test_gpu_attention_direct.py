"""The single-launch decode attention (attention.hip, attn_direct_kernel) against the split kernel and its merge, on the same cache: lengths around the
edges of a batch (128 rows of 128 values, 256 of 64) and behind stale rows, every number of query heads per kv head.

Tolerance: both sum at most 600 products of a softmax in f32 in another order, 600 * 2^-24 = 4e-5 of the largest at worst; logits of two layers, 2e-4."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROWS = (1, 2, 33, 127, 128, 129, 255, 256, 257, 384, 513, 600)


@pytest.mark.parametrize("head_dim,heads,kv_heads", [(64, 8, 8), (64, 8, 4), (64, 8, 2), (64, 8, 1), (128, 4, 4), (128, 4, 2), (128, 4, 1), (128, 8, 1)])
def test_direct_attention_matches_the_split_kernel(pkg, head_dim, heads, kv_heads):
    cfg = pkg.make_config("test-dense", max_seq_len=640, num_heads=heads, num_kv_heads=kv_heads, head_dim=head_dim)
    model = pkg.SynthModel(cfg, mix="Q8_0")
    direct, split = (pkg.HipGpuInference.from_model(model, 640, attn_direct=d) for d in (16, 255))
    prompt = [(7 * i + 5) % cfg.vocab_size for i in range(620)]
    for eng in (direct, split):
        eng.forward_batch(prompt)
    for rows in ROWS:
        got = []
        for eng in (direct, split):
            eng.kv_truncate(rows - 1)
            got.append(eng.forward(rows % cfg.vocab_size))
        assert np.abs(got[0] - got[1]).max() <= 2e-4 * np.abs(got[1]).max(), rows
        for eng in (direct, split):                       # the row that the step overwrote, and the stale ones behind it
            eng.kv_truncate(rows - 1)
            eng.forward_batch(prompt[rows - 1:])
    direct.close()
    split.close()


@pytest.mark.parametrize("bits", [2, 3])
@pytest.mark.parametrize("head_dim,heads,kv_heads", [(64, 8, 8), (64, 8, 1), (128, 4, 2), (128, 8, 1)])
def test_direct_attention_over_codes_matches_the_split_kernel(pkg, head_dim, heads, kv_heads, bits):
    """The same over a TurboQuant cache (attn_tq_direct_kernel): rounds of 128 rows of 128 values, 256 of 64, two ahead.  One layer, so that both
    engines store the same codes (behind a second one a value at a cell's border could fall to either side)."""
    cfg = pkg.make_config("test-dense", max_seq_len=640, num_heads=heads, num_kv_heads=kv_heads, head_dim=head_dim, num_layers=1)
    model = pkg.SynthModel(cfg, mix="Q8_0")
    signs = np.where(np.random.default_rng(3).random(kv_heads * 2 * head_dim) < 0.5, -1.0, 1.0).astype(np.float32)
    kv = {2: pkg.hip_backend.KV_TQ2, 3: pkg.hip_backend.KV_TQ3}[bits]
    direct, split = (pkg.HipGpuInference.from_model(model, 640, attn_direct=d, kv_cache_type=kv, kv_rotation_signs=signs) for d in (16, 255))
    prompt = [(7 * i + 5) % cfg.vocab_size for i in range(620)]
    for eng in (direct, split):
        for t in prompt:
            eng.prefill_token(t)
    for rows in ROWS:
        got = []
        for eng in (direct, split):
            eng.kv_truncate(rows - 1)
            got.append(eng.forward(prompt[rows - 1]))       # (the row that was there)
        assert np.abs(got[0] - got[1]).max() <= 2e-4 * np.abs(got[1]).max(), rows
    direct.close()
    split.close()


@pytest.mark.parametrize("head_dim,heads,kv_heads,limit", [(128, 4, 4, 384), (128, 4, 2, 448), (128, 8, 1, 448), (64, 4, 4, 768), (64, 4, 2, 1152), (64, 8, 2, 1280), (64, 8, 1, 1536)])
def test_the_default_limit_goes_by_the_query_heads_of_a_kv_head(pkg, head_dim, heads, kv_heads, limit):
    """Up to the limit a default engine has the bits of the single launch, behind it those of split and merge."""
    cfg = pkg.make_config("test-dense", max_seq_len=limit + 64, num_heads=heads, num_kv_heads=kv_heads, head_dim=head_dim, num_layers=1)
    model = pkg.SynthModel(cfg, mix="Q8_0")
    engs = [pkg.HipGpuInference.from_model(model, limit + 64, attn_direct=d) for d in (0, 32, 255)]
    prompt = [(7 * i + 5) % cfg.vocab_size for i in range(limit - 1)]
    got = []
    for eng in engs:
        eng.forward_batch(prompt)
        got.append([eng.forward(t) for t in (3, 4)])          # limit and limit + 1 rows
        eng.close()
    assert not np.array_equal(got[1][0], got[2][0]) and not np.array_equal(got[1][1], got[2][1])
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[2][1])
