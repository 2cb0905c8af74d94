"""Which form a batched step's attention takes (engine_batch.hip, short_attn_rows): one launch up to a line that goes by the workgroups it would have and the query heads of a kv head, split and merge behind it.
The last row of the one and the first of the other, for each part of the rule; the logits on both sides are the sequence's own, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,head_dim,sequences,rows", [
    (8, 8, 128, 2, 64), (8, 4, 128, 3, 64), (8, 2, 128, 2, 96), (8, 1, 64, 2, 192),     # fewer than 128 workgroups
    (32, 32, 128, 4, 160), (32, 32, 128, 7, 160), (32, 16, 128, 4, 96), (16, 2, 64, 8, 192),    # fewer than 256
    (32, 32, 128, 8, 256), (32, 32, 64, 12, 320), (32, 16, 128, 8, 512), (32, 8, 128, 8, 640),  # one for every CU
    (32, 32, 128, 16, 128), (32, 16, 64, 16, 512), (32, 8, 128, 16, 512), (64, 64, 64, 16, 128),
])
def test_both_sides_of_the_line(pkg, heads, kv_heads, head_dim, sequences, rows):
    cfg = pkg.make_config("test-dense-d128", max_seq_len=rows + 8, num_heads=heads, num_kv_heads=kv_heads, head_dim=head_dim, num_layers=2, vocab_size=256)
    eng = pkg.HipGpuInference.from_model(pkg.SynthModel(cfg, mix="Q4_K_M"), rows + 8)
    eng.batch_create(sequences)
    tok = np.random.default_rng(rows).integers(0, cfg.vocab_size, rows + 1).astype(np.uint32)
    last = sequences - 1
    eng.batch_prefill(last, tok[:rows - 1])
    eng.forward_batch(tok[:rows - 1])
    for place in (rows - 1, rows):
        eng.set_profiling(True)
        got, _ = eng.forward_multi(list(range(sequences)), [int(tok[place])] * sequences)
        eng.set_profiling(False)
        merges = eng.stats()["kernels"].get("attn_combine", {"launches": 0})["launches"]
        assert merges == (0 if place < rows else 2), place + 1
        assert np.array_equal(got[last].view(np.uint32), eng.forward(int(tok[place])).view(np.uint32)), place + 1
    eng.close()
