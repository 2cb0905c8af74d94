"""A batched step's tokens, positions and slots reach the device in one launch's arguments (engine_batch.hip, stage_control), and only a greedy step moves the positions there: slots in any order and
number, steps with logits, with the arg-max and whole greedy loops in turn, against each sequence alone, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_batch", [1, 3, 16])
def test_steps_of_all_kinds_in_turn(pkg, max_batch):
    cfg = pkg.make_config("test-dense-d128", max_seq_len=48)
    eng = pkg.HipGpuInference.from_model(pkg.SynthModel(cfg, mix="Q4_K_M"), 48)
    eng.batch_create(max_batch)
    rng = np.random.default_rng(max_batch)
    fed, got = [[] for _ in range(max_batch)], [[] for _ in range(max_batch)]   # per slot: tokens fed, (place, logits)
    for kind in ("logits", "greedy", "logits", "loop", "logits", "greedy", "loop", "logits"):
        slots = [int(s) for s in rng.permutation(max_batch)[:int(rng.integers(1, max_batch + 1))]]
        tok = [int(t) for t in rng.integers(0, cfg.vocab_size, len(slots))]
        if kind == "loop":
            out = eng.decode_greedy_multi(slots, tok, 3)
            for i, s in enumerate(slots):
                fed[s] += [tok[i], int(out[0][i]), int(out[1][i])]
        else:
            logits, nxt = eng.forward_multi(slots, tok, greedy=kind == "greedy")
            for i, s in enumerate(slots):
                fed[s].append(tok[i])
                got[s].append((len(fed[s]), logits[i].copy()))
                assert nxt is None or logits[i][nxt[i]] == logits[i].max()
    for s in range(max_batch):
        assert eng.batch_position(s) == len(fed[s])
        eng.reset()
        alone = [eng.forward(t) for t in fed[s]]
        for at, logits in got[s]:
            assert np.array_equal(logits.view(np.uint32), alone[at - 1].view(np.uint32)), (s, at)
    eng.close()


@pytest.mark.parametrize("tokens", [2, 127, 128, 129, 300])
def test_a_slots_prompt_leaves_the_contexts_own_sequence(pkg, tokens):
    """A block's token ids travel in its embedding launch (dequant.hip, embed_block_kernel: 1 to 128 of them), and a slot's prompt does not touch the device's word for the context's own next position:
    the slot against the same prompt of the context's own sequence, and that sequence before and after it, bit for bit."""
    cfg = pkg.make_config("test-dense-d128", max_seq_len=320)
    eng = pkg.HipGpuInference.from_model(pkg.SynthModel(cfg, mix="Q4_K_M"), 320)
    eng.batch_create(2)
    ids = np.random.default_rng(tokens).permutation(cfg.vocab_size)[:tokens].astype(np.uint32)
    ids[-1] = cfg.vocab_size - 1
    eng.forward_batch(ids)
    want = eng.forward(3)
    eng.reset()
    own = [eng.forward(t) for t in (7, 8, 9)]
    eng.reset()
    got = [eng.forward(t) for t in (7, 8)]
    eng.batch_prefill(1, ids)
    got.append(eng.forward(9))
    assert eng.position() == 3 and all(np.array_equal(a.view(np.uint32), b.view(np.uint32)) for a, b in zip(got, own))
    logits, _ = eng.forward_multi([1], [3])
    assert np.array_equal(logits[0].view(np.uint32), want.view(np.uint32))
    eng.close()
