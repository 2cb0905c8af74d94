"""Prompts of 256 tokens (mixtures 160) and more (prefill_wide.hip): the cache they leave, seen through the logits of the tokens that follow, against the exact
engine (f32 throughout, token by token).

Tolerance: that of the 128-token blocks, 1e-2 * max|logit| + 1e-2: the operands of every product are rounded to f16 (2^-12 each) in both paths, and
the rounding of a layer's output is carried on by the next ones; measured 1e-3 to 3e-3 of the largest logit."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _engines(pkg, name, mix, max_seq, **over):
    cfg = pkg.make_config(name, max_seq_len=max_seq, **over)
    model = pkg.SynthModel(cfg, mix=mix, with_bias=bool(over.get("use_neox_rope")))
    return cfg, pkg.HipGpuInference.from_model(model, max_seq, flags=pkg.hip_backend.FLAG_EXACT_PREFILL), pkg.HipGpuInference.from_model(model, max_seq)


def _follow(a, b, toks):
    for t in toks:
        want, got = a.forward(t), b.forward(t)
        assert np.abs(got - want).max() <= 1e-2 * float(np.abs(want).max()) + 1e-2


@pytest.mark.parametrize("name,mix,n,over", [
    ("test-dense", "Q4_K_M", 256, {}), ("test-dense", "Q4_K_M", 257, {}), ("test-dense", "Q5_K_M", 384, {}), ("test-dense", "Q8_0", 511, {}),
    ("test-dense", "Q4_0", 513, {}), ("test-dense", "Q6_K", 641, {}),                       # edges of the 256- and 128-token tiles, every format
    ("test-dense-d128", "Q4_K_M", 300, {}), ("test-dense-d128", "Q5_K_M", 700, dict(use_neox_rope=1)),     # 11 k-blocks; biases and halves
    ("test-dense-d128", "Q4_K_M", 2304, {}),                                                # a full block and a remainder of its own
    ("test-moe", "Q5_K_M", 160, {}), ("test-moe", "Q5_K_M", 259, {}), ("test-moe", "Q4_K_M", 600, {}), ("test-moe", "Q8_0", 400, {})])
def test_long_prompts_match_the_exact_engine(pkg, name, mix, n, over):
    cfg, exact, wide = _engines(pkg, name, mix, n + 16, **over)
    prompt = [(7 * i + 3) % cfg.vocab_size for i in range(n)]
    for eng in (exact, wide):
        eng.forward_batch(prompt)
        assert eng.position() == n
    _follow(exact, wide, (5, 77, 9))
    wide.reset()                                             # the same prompt again: bit for bit
    wide.forward_batch(prompt)
    first = wide.forward(5)
    wide.reset()
    wide.forward_batch(prompt)
    assert np.array_equal(wide.forward(5), first)
    exact.close()
    wide.close()


def test_long_prompts_continue_a_sequence_and_fill_slots(pkg):
    cfg, exact, wide = _engines(pkg, "test-dense", "Q4_K_M", 700)
    a, b = [(5 * i + 1) % cfg.vocab_size for i in range(37)], [(11 * i + 2) % cfg.vocab_size for i in range(419)]
    for eng in (exact, wide):
        eng.forward_batch(a)
        eng.forward(77)
        eng.forward_batch(b)
        assert eng.position() == 457
    _follow(exact, wide, (3, 4))
    wide.batch_create(3)
    wide.batch_prefill(2, b)
    exact.reset()
    exact.forward_batch(b)
    want, got = exact.forward(8), wide.forward_multi([2], [8])[0][0]
    assert np.abs(got - want).max() <= 1e-2 * float(np.abs(want).max()) + 1e-2
    assert wide.position() == 459    # the context's own sequence is where it was
    exact.close()
    wide.close()


def test_long_prompts_without_their_own_memory_take_the_short_blocks(pkg):
    """An allocation that fails, whichever it is, is not left half made and costs speed alone; with the memory back the long path is taken.  Its copy of a layer's cache
    follows the positions in use, not the context's capacity."""
    cfg = pkg.make_config("test-dense", max_seq_len=65536)
    model = pkg.SynthModel(cfg, mix="Q4_K_M")
    eng, whole, short = (pkg.HipGpuInference.from_model(model, 65536) for _ in range(3))
    prompt = [(7 * i + 3) % cfg.vocab_size for i in range(300)]
    for at in range(0, 300, 100):
        short.forward_batch(prompt[at:at + 100])             # blocks of 100 tokens
    want = short.forward(9)
    for e in (eng, whole):
        e.forward_batch(prompt[:100])
    before = eng.stats()["scratch_bytes"]
    whole.forward_batch(prompt)
    full = whole.stats()["scratch_bytes"]
    copy = cfg.num_kv_heads * 4096 * cfg.head_dim * 2 * 6     # K and V of 4096 rows in three numbers of two bytes
    assert before + copy < full
    for nth in range(1, 40):
        eng.reset()
        eng.debug_fail_alloc(nth)
        eng.forward_batch(prompt)
        assert eng.position() == 300
        got = eng.forward(9)
        assert np.abs(got - want).max() <= 1e-2 * float(np.abs(want).max()) + 1e-2, nth
        held = eng.stats()["scratch_bytes"]
        if held == full:
            break
        assert held in (before, full - copy), nth              # (the copy comes last; the others wait for it)
    assert nth > 3 and held == full
    eng.debug_fail_alloc(0)
    eng.forward_batch(prompt)                                 # 301 .. 600: grows nothing
    assert eng.stats()["scratch_bytes"] == full
    tail = [(5 * i) % cfg.vocab_size for i in range(4000)]
    eng.debug_fail_alloc(1)
    eng.forward_batch(tail)                                   # behind position 4096: no room
    assert eng.stats()["scratch_bytes"] == full - copy
    eng.forward_batch(tail)                                   # 4601 .. 8600: rows of 12288
    assert eng.stats()["scratch_bytes"] == full + 2 * copy and eng.position() == 301 + 300 + 8000
    exact = pkg.HipGpuInference.from_model(model, 65536, flags=pkg.hip_backend.FLAG_EXACT_PREFILL)
    exact.forward_batch(prompt)
    eng.reset()
    eng.forward_batch(prompt)
    _follow(exact, eng, (5, 77))
    for e in (eng, whole, short, exact):
        e.close()


@pytest.mark.parametrize("name,mix,n", [("test-dense", "Q4_K_M", 385), ("test-dense", "Q8_0", 448), ("test-dense", "Q6_K", 449), ("test-dense", "Q4_0", 704), ("test-dense", "Q5_K_M", 420),
                                        ("test-moe", "Q5_K_M", 290), ("test-moe", "Q6_K", 350), ("test-moe", "Q4_0", 330), ("test-moe", "Q4_K_M", 384)])
def test_last_tiles_of_up_to_192_tokens(pkg, name, mix, n):
    """The body for 129 to 192 tokens: a last tile's first, last and first beyond its range, experts whose rows fall into it (four of them, two a token).  A token's sums are the same in a tile of any
    size, so the cache is, bit for bit, what the same tokens leave as part of a prompt whose last tile is full."""
    full = (n + 255) // 256 * 256
    cfg = pkg.make_config(name, max_seq_len=full + 16)
    model = pkg.SynthModel(cfg, mix=mix)
    a, b = (pkg.HipGpuInference.from_model(model, full + 16) for _ in range(2))
    prompt = [(7 * i + 3) % cfg.vocab_size for i in range(full)]
    a.forward_batch(prompt[:n])
    b.forward_batch(prompt)
    b.kv_truncate(n)
    for t in (5, 77, 9):
        assert np.array_equal(a.forward(t), b.forward(t))


@pytest.mark.parametrize("n", [200, 300])
def test_stages_against_one_context(pkg, n):
    """Stages hand blocks of 128 tokens over: below 256 tokens the bits of a single context, which takes the long path from there on, behind it its rounding."""
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]

    def hop(dst, src, rows):
        s0.synchronize()
        assert hip.hipMemcpy(dst, src, rows * cfg.hidden_size * 4, 3) == 0 and hip.hipDeviceSynchronize() == 0

    cfg = pkg.make_config("test-dense-d128", max_seq_len=400)
    model = pkg.SynthModel(cfg, mix="Q4_K_M")
    one, s0, s1 = (pkg.HipGpuInference.from_model(model, 400, layer_range=r) for r in (None, (0, 1), (1, cfg.num_layers)))
    prompt = [(7 * i + 3) % cfg.vocab_size for i in range(n)]
    one.forward_batch(prompt)
    for at in range(0, n, 128):
        block = prompt[at:at + 128]
        s0.stage_prefill_batch(block, len(block))
        hop(s1.stage_hidden_block_ptr(), s0.stage_hidden_block_ptr(), len(block))
        s1.stage_prefill_batch(None, len(block))
        s1.synchronize()
    want = one.forward(5)
    s0.stage_forward(5)
    hop(s1.stage_hidden_ptr(), s0.stage_hidden_ptr(), 1)
    got = s1.stage_forward(0, want_logits=True)
    assert n >= 256 or np.array_equal(want, got)
    assert np.abs(got - want).max() <= 1e-2 * float(np.abs(want).max()) + 1e-2
    for e in (one, s0, s1):
        e.close()
