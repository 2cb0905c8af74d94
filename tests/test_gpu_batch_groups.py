"""The batched step's mat-vec from three sequences on takes them in groups (matvec_batch.hip: of four on the integer matrix cores, from five
sequences on of eight on the bf16 ones, 8-bit weights apart): group sizes around full ones, every weight format, plans with whole rows per
workgroup and plans with k-slices.

Per (row, sequence) the kernel does the single-sequence kernel's floating-point operations in its order, on sums that are exact, so the
bound is equality of all bits with a single-sequence engine that runs the split attention too (attn_direct=255)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,mix,sizes,kw", [
    ("test-dense-d128", "Q4_K_M", (3, 4, 5, 7, 8, 9, 12, 13, 16), {}),
    ("test-dense-d128", "Q5_K_M", (3, 6, 11, 15), {}),
    ("test-dense-d128", "Q6_K", (3, 5, 10, 14), {}),
    ("test-dense-d128", "Q8_0", (3, 5, 9, 16), {}),
    ("test-dense-d128", "Q4_0", (3, 5, 9, 16), {}),
    ("llama-3-8b", "Q4_K_M", (3, 8, 13), dict(num_layers=1, vocab_size=4096)),     # gate | up: whole rows per workgroup
    ("llama-3-8b", "Q5_K_M", (5, 16), dict(num_layers=1, vocab_size=4096)),
])
def test_groups_of_sequences_are_bitwise_the_single_sequence(pkg, name, mix, sizes, kw):
    cfg = pkg.make_config(name, max_seq_len=32, **kw)
    model = pkg.SynthModel(cfg, mix=mix)
    multi = pkg.HipGpuInference.from_model(model, 32)
    single = pkg.HipGpuInference.from_model(model, 32, attn_direct=255)
    multi.batch_create(16)
    tok = np.random.default_rng(5).integers(0, cfg.vocab_size, (16, 2))
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


@pytest.mark.parametrize("name,max_seq", [("test-dense-d128", 640), ("test-dense-d128", 2100), ("test-dense", 500)])
def test_splits_walked_by_one_workgroup_are_bitwise_the_single_sequence(pkg, name, max_seq):
    """The batched attention gives a workgroup several splits, with and without rows: contexts around the rows a split takes at a time."""
    cfg = pkg.make_config(name, max_seq_len=max_seq)
    model = pkg.SynthModel(cfg, mix="Q4_K_M")
    multi = pkg.HipGpuInference.from_model(model, max_seq)
    single = pkg.HipGpuInference.from_model(model, max_seq, attn_direct=255)
    lens = (2, 3, 7, 8, 9, 16, 17, 63, 64, 65, 127, 256, 257, 300, 449, 480)
    multi.batch_create(16)
    tok = np.random.default_rng(8).integers(0, cfg.vocab_size, (16, max(lens) + 2))
    for s, n in enumerate(lens):
        multi.batch_prefill(s, tok[s, :n])
    got = [multi.forward_multi(list(range(16)), [int(tok[s, n + k]) for s, n in enumerate(lens)])[0] for k in range(2)]
    for s, n in enumerate(lens):
        single.reset()
        single.forward_batch(tok[s, :n])
        for k in range(2):
            want = single.forward(int(tok[s, n + k]))
            assert np.array_equal(got[k][s].view(np.uint32), want.view(np.uint32)), (s, k)
    multi.close()
    single.close()


def test_sums_at_the_edge_of_their_range_are_bitwise_the_single_sequence(pkg):
    """Six-bit weights near 63 on chunks whose low 16 bits are near their extremes and all of one sign: the sum over a chunk's low halves (16 * 63 * 32896) needs 25 bits,
    and the large value that sets the chunk's scale meets a weight of zero, so that the sum is all there is of the product."""
    syn = pkg.synth

    class Model(pkg.SynthModel):
        def specs(self, layers=None):
            for s in super().specs(layers):
                yield syn.TensorSpec(s.name, syn.F32, s.ne) if s.name == "token_embd.weight" else s

    cfg = pkg.make_config("test-dense-d128", max_seq_len=8, num_layers=1)
    model, rng = Model(cfg, mix="Q6_K"), np.random.default_rng(4)
    k, vocab = cfg.hidden_size, cfg.vocab_size
    x = rng.integers(32640, 32768, (vocab, k // 16, 16))
    x[::2] = -rng.integers(32769, 32897, x[::2].shape)                 # digits -128, < 0
    x = x.astype(np.float32) * np.float32(2.0 ** -29)
    x[..., 3] = 1.0
    model._cache["token_embd.weight"] = x.reshape(-1).view(np.uint8)
    model._cache["blk.0.attn_norm.weight"] = np.ones(k, dtype=np.float32).view(np.uint8)
    for name, n in (("attn_q", cfg.num_heads * cfg.head_dim), ("attn_k", cfg.num_kv_heads * cfg.head_dim), ("attn_v", cfg.num_kv_heads * cfg.head_dim)):
        q = rng.integers(56, 64, (n * k // 256, 256))
        q[:, 3::16] = 0
        ql, qh = np.zeros((len(q), 128), np.uint8), np.zeros((len(q), 64), np.uint8)
        for half in range(2):                                          # block_q6_K: 128 values a half, four stripes of 32
            for stripe in range(4):
                v = q[:, half * 128 + stripe * 32:half * 128 + stripe * 32 + 32]
                ql[:, half * 64 + stripe % 2 * 32:half * 64 + stripe % 2 * 32 + 32] |= ((v & 15) << (4 * (stripe // 2))).astype(np.uint8)
                qh[:, half * 32:half * 32 + 32] |= ((v >> 4) << (2 * stripe)).astype(np.uint8)
        sc = rng.integers(1, 64, (len(q), 16)).astype(np.int8).view(np.uint8)
        d = np.full((len(q), 1), 0.01, np.float16).view(np.uint8)
        model._cache[f"blk.0.{name}.weight"] = np.concatenate([ql, qh, sc, d], axis=1).reshape(-1)
    multi = pkg.HipGpuInference.from_model(model, 8)
    single = pkg.HipGpuInference.from_model(model, 8, attn_direct=255)
    multi.batch_create(16)
    for n in (2, 4, 5, 9, 16):
        for s in range(16):
            multi.batch_reset(s)
        tok = rng.integers(0, vocab, 16)
        got, _ = multi.forward_multi(list(range(n)), tok[:n])
        for s in range(n):
            single.reset()
            assert np.array_equal(got[s].view(np.uint32), single.forward(int(tok[s])).view(np.uint32)), (n, s)
    multi.close()
    single.close()


@pytest.mark.parametrize("max_batch,sizes", [(16, 7), (12, 6), (4, 4), (2, 2), (1, 1)])
def test_creating_slots_runs_every_group_size_outside_a_capture(pkg, max_batch, sizes):
    """A kernel first launched inside a capture may be left out of its replays: lgh_batch_create launches those of steps of 1, 2, 3, 4, 5, 9 and 13 sequences, which between
    them are all, before any graph is made.  (One output projection a step.)"""
    cfg = pkg.make_config("test-dense-d128", max_seq_len=16)
    eng = pkg.HipGpuInference.from_model(pkg.SynthModel(cfg, mix="Q4_K_M"), 16)
    eng.set_profiling(True)
    eng.batch_create(max_batch)
    eng.forward_multi([0], [1])                               # (reads the events of all launches so far)
    assert eng.stats()["kernels"]["output"]["launches"] == sizes + 1
    assert all(eng.batch_position(s) == (s == 0) for s in range(max_batch))
    eng.close()
