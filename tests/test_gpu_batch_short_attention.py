"""The batched step's attention in one launch (attention.hip, attn_multi_direct_kernel) against split and merge, which a context with slots uses for its own sequence: all bits equal.  Lengths around a
split's rows (8 or 16 of 128 values), a round of the workgroup, the rows behind which a split takes a second step (256, 512) and the lines up to which the launch is taken; splits of four and of eight waves
(capacities below 2048 and from there on); sequences of very different lengths in one step.  (Prompts of 0 or of 2 and more tokens: lgh_prefill_batch feeds a
single one through the exact step, lgh_batch_prefill through a prompt block, whose products have 16-bit operands.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,head_dim,max_seq,lens", [
    (8, 2, 128, 300, (0, 2, 6, 7, 8, 30, 31, 32, 100, 125)),                     # up to 128 rows with fewer than 128 workgroups
    (8, 2, 64, 300, (2, 14, 15, 16, 63, 64, 130, 253)),                          # 256 rows of 64
    (8, 4, 128, 300, (2, 15, 33, 126)),
    (8, 1, 128, 2100, (3, 14, 15, 16, 17, 31, 124, 125)),                        # eight waves a split
    (16, 2, 128, 600, (2, 40, 127, 128, 200, 250, 252, 253)),                    # 256 rows with 128 workgroups or more
    (32, 8, 128, 900, (5, 255, 256, 257, 300, 511, 512, 700)),                   # 768 rows with 256 or more
    (32, 8, 64, 2100, (9, 600, 1022, 1024, 1030, 31, 500, 1300)),
    (32, 32, 128, 2100, (2, 500, 512, 513, 600, 40, 200, 760)),
])
def test_one_launch_equals_split_and_merge(pkg, heads, kv_heads, head_dim, max_seq, lens):
    cfg = pkg.make_config("test-dense-d128", max_seq_len=max_seq, num_heads=heads, num_kv_heads=kv_heads, head_dim=head_dim, num_layers=2, vocab_size=512)
    eng = pkg.HipGpuInference.from_model(pkg.SynthModel(cfg, mix="Q4_K_M"), max_seq)
    steps = 3
    tok = np.random.default_rng(heads + max_seq).integers(0, cfg.vocab_size, (len(lens), max(lens) + steps))
    eng.batch_create(len(lens))
    for s, n in enumerate(lens):
        if n:
            eng.batch_prefill(s, tok[s, :n])
    got = [eng.forward_multi(list(range(len(lens))), [int(tok[s, n + k]) for s, n in enumerate(lens)])[0] for k in range(steps)]
    for s, n in enumerate(lens):
        eng.reset()
        if n:
            eng.forward_batch(tok[s, :n])
        for k in range(steps):
            want = eng.forward(int(tok[s, n + k]))
            assert np.array_equal(got[k][s].view(np.uint32), want.view(np.uint32)), (n + k + 1, float(np.abs(got[k][s] - want).max()))
    eng.close()


def test_a_greedy_loop_across_the_line(pkg):
    """decode_greedy_multi walks past the line (96 rows here): the launches change between two steps, the tokens are the single steps'."""
    cfg = pkg.make_config("test-dense-d128", max_seq_len=300, num_layers=2)
    eng = pkg.HipGpuInference.from_model(pkg.SynthModel(cfg, mix="Q4_K_M"), 300)
    eng.batch_create(2)
    tok = np.random.default_rng(3).integers(0, cfg.vocab_size, (2, 92))
    for s in range(2):
        eng.batch_prefill(s, tok[s])
    loop = eng.decode_greedy_multi([0, 1], [5, 9], 8)
    for s in range(2):
        eng.batch_reset(s)
        eng.batch_prefill(s, tok[s])
    cur, want = [5, 9], []
    for _ in range(8):
        _, cur = eng.forward_multi([0, 1], [int(t) for t in cur], want_logits=True, greedy=True)
        want.append(list(cur))
    assert np.array_equal(np.asarray(loop), np.asarray(want))
    eng.close()
