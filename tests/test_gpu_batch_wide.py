"""The wide images of a batched step's vectors (xq.h), from five sequences on: left by whoever writes the vector (embedding, attention in one launch and in two, over f32 slots and over codes, the mat-vecs' epilogues, the
mixtures' sum), or made from the digits where nobody did (a mixture that goes sequence by sequence).  Slots as many as sequences, so that the last block's transfers end behind the last record; group sizes around full ones.

The kernel does the single-sequence kernel's operations on the same numbers: equality of all bits with the context's own sequence, which takes the attention that its slots take."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,mix,B,kv,cap", [
    ("test-dense-d128", "Q4_K_M", 5, None, 96), ("test-dense-d128", "Q5_K_M", 9, None, 2304), ("test-dense", "Q4_0", 13, None, 96),
    ("test-dense-d128", "Q4_K_M", 7, "tq3", 96), ("test-dense", "Q5_K_M", 6, "tq2-qjl", 96), ("test-dense-d128", "Q4_0", 8, "tq3", 9000),
    ("test-moe", "Q4_K_M", 6, None, 96), ("test-moe-grouped", "Q5_K_M", 11, None, 96),
])
def test_steps_from_wide_images_are_bitwise_the_single_sequence(pkg, name, mix, B, kv, cap):
    hb = pkg.hip_backend
    over = {}
    if name == "test-moe-grouped":
        name, over = "test-moe", dict(expert_intermediate_size=1024)
    cfg = pkg.make_config(name, max_seq_len=cap, **over)
    model = pkg.SynthModel(cfg, mix=mix)
    opt = {}
    if kv:
        rng = np.random.default_rng(29)
        n = cfg.num_layers * cfg.num_kv_heads * cfg.head_dim
        opt = dict(kv_cache_type={"tq3": hb.KV_TQ3, "tq2-qjl": hb.KV_TQ2_QJL}[kv], kv_rotation_signs=np.where(rng.integers(0, 2, 2 * n) == 1, 1.0, -1.0).astype(np.float32))
        if kv.endswith("qjl"):
            opt["kv_qjl_matrices"] = rng.standard_normal(n * cfg.head_dim).astype(np.float32)
    multi = pkg.HipGpuInference.from_model(model, cap, **opt)
    multi.batch_create(B)
    tok = np.random.default_rng(3).integers(0, cfg.vocab_size, (B, 3))
    got = [multi.forward_multi(list(range(B)), tok[:, step])[0].copy() for step in range(3)]
    for s in range(B):
        multi.reset()
        for step in range(3):
            want = multi.forward(int(tok[s, step]))
            assert np.array_equal(got[step][s].view(np.uint32), want.view(np.uint32)), (s, step)
    multi.close()
