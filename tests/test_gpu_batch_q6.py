"""Six-bit weights in a batched step, from five sequences on one digit a row on the bf16 matrix cores (matvec_batch.hip, mvqb8): alone with whole rows per workgroup and with k-slices, and beside four- and five-bit ones in one launch, whose workgroups walk all of k there too (24576 rows of Q, K and V).  Group sizes
of every instantiation.

The sums and their roundings are the single-sequence kernel's: equality of all bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,mix,sizes,kw", [
    ("llama-3-8b", "Q6_K", (5, 12, 16), dict(num_layers=1, vocab_size=4096)),
    ("test-dense-d128", "Q6_K", (8, 9, 13), dict(num_layers=2, vocab_size=21000)),
    ("test-dense-d128", "Q4_K_M", (5, 9, 16), dict(num_layers=2, hidden_size=1024, num_heads=128, num_kv_heads=32, intermediate_size=1024, vocab_size=1000)),
    ("test-dense-d128", "Q5_K_M", (8, 11, 14), dict(num_layers=2, hidden_size=1024, num_heads=128, num_kv_heads=32, intermediate_size=1024, vocab_size=1000)),
])
def test_six_bits_are_bitwise_the_single_sequence(pkg, name, mix, sizes, kw):
    cfg = pkg.make_config(name, max_seq_len=16, **kw)
    model = pkg.SynthModel(cfg, mix=mix)
    multi = pkg.HipGpuInference.from_model(model, 16)
    single = pkg.HipGpuInference.from_model(model, 16, attn_direct=255)
    multi.batch_create(16)
    tok = np.random.default_rng(23).integers(0, cfg.vocab_size, (16, 2))
    want = []
    for s in range(16):
        single.reset()
        want.append([single.forward(int(t)).copy() for t in tok[s]])
    for n in sizes:
        for s in range(16):
            multi.batch_reset(s)
        for step in range(2):
            got, _ = multi.forward_multi(list(range(n)), tok[:n, step])
            for s in range(n):
                assert np.array_equal(got[s].view(np.uint32), want[s][step].view(np.uint32)), (n, s, step)
    multi.close()
    single.close()
