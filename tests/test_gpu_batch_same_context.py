"""A batched sequence and lgh_forward on the context that holds the slots, default flags: the same bits at every length (include/llama_gguf_hip.h), over f32 and
TurboQuant caches, in contexts whose capacity lies on either side of the single-launch attention's limit (1152 rows at head size 128)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _same(eng, cfg, lens, steps, feed):
    """Slots with prompts of `lens` tokens, `steps` more in the batch; the context's own sequence with each history in turn."""
    rng = np.random.default_rng(len(lens) + max(lens))
    tok = rng.integers(0, cfg.vocab_size, (len(lens), max(lens) + steps))
    eng.batch_create(len(lens))
    for s, n in enumerate(lens):
        eng.batch_prefill(s, tok[s, :n])
    got = [eng.forward_multi(list(range(len(lens))), [int(tok[s, n + k]) for s, n in enumerate(lens)])[0] for k in range(steps)]
    for s, n in enumerate(lens):
        eng.reset()
        feed(eng, tok[s, :n])
        for k in range(steps):
            want = eng.forward(int(tok[s, n + k]))
            assert np.array_equal(got[k][s].view(np.uint32), want.view(np.uint32)), (lens[s] + k + 1, float(np.abs(got[k][s] - want).max()))


@pytest.mark.parametrize("name,max_seq", [("test-dense-d128", 500), ("test-dense", 640)])
def test_f32_slots(pkg, name, max_seq):
    cfg = pkg.make_config(name, max_seq_len=max_seq)
    eng = pkg.HipGpuInference.from_model(pkg.SynthModel(cfg, mix="Q4_K_M"), max_seq)
    _same(eng, cfg, (2, 20, 62, 63, 64, 127, 255, 446, 447), 3, lambda e, t: e.forward_batch(t))
    eng.close()


def _one_by_one(eng, tokens):
    for t in tokens:
        eng.prefill_token(int(t))


@pytest.mark.parametrize("name,max_seq,direct", [("test-dense-d128", 300, 0), ("test-dense-d128", 2048, 0), ("test-dense", 300, 0),
                                                 ("test-dense-d128", 300, 255), ("test-dense", 300, 255)])
@pytest.mark.parametrize("bits", [2, 3])
def test_turboquant_slots(pkg, name, max_seq, direct, bits):
    """Single-launch (capacity within the limit, rounds of 128 and 256 rows), split and merge (beyond it, or asked for)."""
    cfg = pkg.make_config(name, max_seq_len=max_seq)
    signs = np.where(np.random.default_rng(5).random(cfg.num_layers * cfg.num_kv_heads * 2 * cfg.head_dim) < 0.5, -1.0, 1.0).astype(np.float32)
    kv = {2: pkg.hip_backend.KV_TQ2, 3: pkg.hip_backend.KV_TQ3}[bits]
    eng = pkg.HipGpuInference.from_model(pkg.SynthModel(cfg, mix="Q4_K_M"), max_seq, attn_direct=direct, kv_cache_type=kv, kv_rotation_signs=signs)
    _same(eng, cfg, (3, 126, 127, 128, 255, 257), 3, _one_by_one)
    eng.close()
