"""The launch that adds up a batched step's partial sums (matvec_batch.hip, mvqb_rows_kernel): four k-slices and eight, some of them empty, four row tiles a workgroup, more rows x sequences than threads, a norm over more than
256 chunks, Q, K and V of sizes that share no power of two, the residual with and without the next norm.

Sums and epilogue are the single-sequence kernel's operations in its order: equality of all bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mix,kw", [
    ("Q4_K_M", dict(hidden_size=1024, num_heads=8, num_kv_heads=4, intermediate_size=8704)),     # four slices; gate | up split over k, four tiles a workgroup
    ("Q8_0", dict(hidden_size=4864, num_heads=38, num_kv_heads=19, intermediate_size=1024)),     # slices of unequal size, 304 chunks
    ("Q4_0", dict(hidden_size=2816, num_heads=22, num_kv_heads=11, intermediate_size=2304)),     # eleven and nine blocks
])
def test_rows_are_bitwise_the_single_sequence(pkg, mix, kw):
    cfg = pkg.make_config("test-dense-d128", max_seq_len=16, num_layers=2, vocab_size=1000, **kw)
    model = pkg.SynthModel(cfg, mix=mix)
    multi = pkg.HipGpuInference.from_model(model, 16)
    single = pkg.HipGpuInference.from_model(model, 16, attn_direct=255)
    multi.batch_create(16)
    tok = np.random.default_rng(11).integers(0, cfg.vocab_size, (16, 2))
    want = []
    for s in range(16):
        single.reset()
        want.append([single.forward(int(t)).copy() for t in tok[s]])
    for n in (2, 3, 5, 9, 16):
        for s in range(16):
            multi.batch_reset(s)
        for step in range(2):
            got, _ = multi.forward_multi(list(range(n)), tok[:n, step])
            for s in range(n):
                assert np.array_equal(got[s].view(np.uint32), want[s][step].view(np.uint32)), (n, s, step)
    multi.close()
    single.close()
