"""The token behind a prompt block, whose step runs beside the block (engine.hip, tail_layer), against the block and then the step: all bits equal, its own logits and those of the tokens after it.  Portions
around one block (128 tokens) and a remainder of one token, from nothing and behind earlier tokens, several wanted places, short and long contexts (the two forms of attention), mixtures, a context with slots."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model,mix,max_seq,slots", [
    ("test-dense", "Q4_K_M", 700, 0),
    ("test-dense-d128", "Q8_0", 700, 0),
    ("test-dense-d128", "Q5_K_M", 5000, 2),
    ("test-moe", "Q5_K_M", 700, 0),
])
def test_a_step_beside_its_block(pkg, model, mix, max_seq, slots):
    cfg = pkg.make_config(model, max_seq_len=max_seq, hidden_size=2048, num_layers=2)   # (narrower models take it from more tokens on)
    m = pkg.SynthModel(cfg, mix=mix)
    beside, behind = (pkg.HipGpuInference.from_model(m, max_seq) for _ in range(2))
    assert beside.prefill_is_batched()
    if not beside.beside_blocks()[0]:
        pytest.skip("no stream here runs beside the context's own")
    ran = 0
    if slots:
        beside.batch_create(slots)
        behind.batch_create(slots)
    tok = np.random.default_rng(5).integers(0, cfg.vocab_size, 700).astype(np.uint32)
    for before, portion in ((0, (3,)), (0, (17,)), (0, (129,)), (0, (130,)), (5, (64, 3, 1, 130)), (0, (258,)), (0, (300, 40)), (160, (150,))):
        beside.reset()
        behind.reset()
        if before:
            beside.forward_batch(tok[:before])
            behind.forward_batch(tok[:before])
        n = sum(portion)
        got = beside.eval(tok[before:before + n], [int(v) - 1 for v in np.cumsum(portion)])
        ran += sum(length > 2 for length in portion)   # two tokens in front and more: a block
        at = before
        for i, length in enumerate(portion):
            if length > 1:
                behind.forward_batch(tok[at:at + length - 1])
            want = behind.forward(int(tok[at + length - 1]))
            at += length
            assert np.array_equal(got[i].view(np.uint32), want.view(np.uint32)), (before, portion, i)
        assert beside.position() == behind.position() == at
        for t in (4, 9):
            assert np.array_equal(beside.forward(t).view(np.uint32), behind.forward(t).view(np.uint32)), (before, portion)
    assert ran // 2 < beside.beside_blocks()[1] <= ran     # (one whose stream was not idle at once goes behind its block)
    assert behind.beside_blocks()[1] == 0
    beside.close()
    behind.close()


def test_large_blocks_go_first(pkg):
    """1536 tokens of width 4096 and fewer have the step beside them, larger blocks in front of it."""
    cfg = pkg.make_config("test-dense-d128", max_seq_len=1700, hidden_size=4096, intermediate_size=512, num_heads=32, num_kv_heads=8, num_layers=2, vocab_size=512)
    m = pkg.SynthModel(cfg, mix="Q8_0")
    beside, behind = (pkg.HipGpuInference.from_model(m, 1700) for _ in range(2))
    if not beside.beside_blocks()[0]:
        pytest.skip("no stream here runs beside the context's own")
    tok = np.random.default_rng(6).integers(0, cfg.vocab_size, 1700).astype(np.uint32)
    for block, goes in ((1536, True), (1537, False), (1600, False), (700, True)):
        for attempt in range(5):                  # (one whose stream was not idle at once goes behind its block)
            beside.reset()
            before = beside.beside_blocks()[1]
            got = beside.eval(tok[:block + 1], [block])[0]
            if beside.beside_blocks()[1] > before:
                break
        assert (beside.beside_blocks()[1] > before) == goes, block
        behind.reset()
        behind.forward_batch(tok[:block])
        assert np.array_equal(got.view(np.uint32), behind.forward(int(tok[block])).view(np.uint32)), block
        assert np.array_equal(beside.forward(4).view(np.uint32), behind.forward(4).view(np.uint32)), block
    beside.close()
    behind.close()


def test_narrow_models_from_more_tokens_on(pkg):
    """A model of width 1024: stretches of 48 tokens and more have the step beside their block, shorter ones in front of it."""
    cfg = pkg.make_config("test-dense", max_seq_len=300, hidden_size=1024, num_layers=2)
    m = pkg.SynthModel(cfg, mix="Q4_K_M")
    beside, behind = (pkg.HipGpuInference.from_model(m, 300) for _ in range(2))
    if not beside.beside_blocks()[0]:
        pytest.skip("no stream here runs beside the context's own")
    tok = np.random.default_rng(8).integers(0, cfg.vocab_size, 300).astype(np.uint32)
    for block, goes in ((2, False), (47, False), (48, True), (128, True), (131, True)):
        for attempt in range(5):
            beside.reset()
            before = beside.beside_blocks()[1]
            got = beside.eval(tok[:block + 1], [block])[0]
            if beside.beside_blocks()[1] > before:
                break
        assert (beside.beside_blocks()[1] > before) == goes, block
        behind.reset()
        behind.forward_batch(tok[:block])
        assert np.array_equal(got.view(np.uint32), behind.forward(int(tok[block])).view(np.uint32)), block
    beside.close()
    behind.close()


def test_the_step_behind_a_first_prompt_is_there(pkg):
    """A prompt's last token is launched kernel by kernel where it runs beside its block; the graph that the tokens after it take is captured in the same call, not in theirs."""
    m = pkg.SynthModel(pkg.make_config("test-dense", max_seq_len=300, hidden_size=2048, num_layers=2), mix="Q4_K_M")
    eng = pkg.HipGpuInference.from_model(m, 300)
    assert eng.stats()["graph_nodes"] == 0
    eng.eval(np.arange(40) % m.config.vocab_size, [39])
    nodes = eng.stats()["graph_nodes"]
    assert nodes > 0
    eng.forward(3)
    assert eng.stats()["graph_nodes"] == nodes
    eng.close()


def test_work_on_the_null_stream_sends_the_step_behind(pkg):
    """The stream shares the null stream's queue: while others' work is in it, a step goes behind its block and waits for none of that."""
    m = pkg.SynthModel(pkg.make_config("test-dense", max_seq_len=200, hidden_size=2048, num_layers=2), mix="Q4_K_M")
    eng = pkg.HipGpuInference.from_model(m, 200)
    if not eng.beside_blocks()[0]:
        pytest.skip("no stream here runs beside the context's own")
    tok = np.arange(150) * 7 % m.config.vocab_size
    want = eng.eval(tok, [149])[0]
    hip, big, words = C.CDLL(pkg.hip_backend.load_library()._name), C.c_void_p(), 1 << 28   # (the same library: its runtime's functions are found through it)
    assert hip.hipMalloc(C.byref(big), C.c_size_t(words * 4)) == 0
    for _ in range(3):
        eng.reset()
        before = eng.beside_blocks()[1]
        for k in range(50):                       # some 0.2 ms each
            assert hip.hipMemsetD32Async(big, k, C.c_size_t(words), None) == 0
        got = eng.eval(tok, [149])[0]
        assert eng.beside_blocks()[1] == before
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        assert hip.hipStreamSynchronize(None) == 0
    assert hip.hipFree(big) == 0
    eng.close()


def test_contexts_at_work_share_one_stream(pkg):
    """The device has one stream for such steps, taken by one prompt at a time and only while no other is at work: contexts in threads give what each gives alone, and contexts come and go around it."""
    m = pkg.SynthModel(pkg.make_config("test-dense-d128", max_seq_len=400, hidden_size=2048, num_layers=2), mix="Q4_K_M")
    tok = np.random.default_rng(7).integers(0, m.config.vocab_size, 400).astype(np.uint32)
    lengths = (3, 40, 129, 300)
    first = pkg.HipGpuInference.from_model(m, 400)
    want = {}
    for n in lengths:
        first.reset()
        want[n] = first.eval(tok[:n], [n - 1])[0].copy()
    at_work = [first] + [pkg.HipGpuInference.from_model(m, 400) for _ in range(3)]
    before = [e.beside_blocks()[1] for e in at_work]
    wrong = []

    def prompts(e, k):
        for i in range(24):
            n = lengths[(i + k) % 4]
            e.reset()
            if not np.array_equal(e.eval(tok[:n], [n - 1])[0].view(np.uint32), want[n].view(np.uint32)):
                wrong.append((k, i, n))
    for _ in range(2):
        threads = [threading.Thread(target=prompts, args=(e, k)) for k, e in enumerate(at_work)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong
        ran = [e.beside_blocks()[1] - b for e, b in zip(at_work, before)]
        assert sum(ran) < 24 * len(at_work), "every prompt had the device to itself"
        at_work.pop(0).close()                    # the context that made the stream goes first
        before.pop(0)
        before = [e.beside_blocks()[1] for e in at_work]
    for e in at_work:
        e.close()
    again = pkg.HipGpuInference.from_model(m, 400)
    assert np.array_equal(again.eval(tok[:40], [39])[0].view(np.uint32), want[40].view(np.uint32))
    again.close()
