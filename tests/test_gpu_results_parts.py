"""Results on their way to the caller (engine.hip: results_take): parts of 16 384 floats that the device answers one by one, 32 of them a launch, halves in turn for more.  Sizes around a part and around all of them; rows
that do not lie one behind the other; the results a step brings itself against those of a call of their own; many calls one after the other (every launch has a number)."""
import numpy as np
import pytest

import layered_cases as lc

pytestmark = pytest.mark.gpu
PART = 16384


@pytest.mark.parametrize("vocab", [PART - 1, PART, PART + 1, 3 * PART, 32 * PART - 1, 32 * PART, 32 * PART + 1, 40 * PART + 77])
def test_logits_a_step_brings_are_those_read_behind_it(pkg, vocab):
    cfg = pkg.make_config("test-dense", max_seq_len=24, vocab_size=vocab, num_layers=1)
    eng = pkg.HipGpuInference.from_model(pkg.SynthModel(cfg, mix="Q8_0"), 24)
    lib = pkg.hip_backend.load_library()
    for i in range(20):
        got = eng.forward((97 * i) % vocab)
        again = np.full(vocab, np.nan, np.float32)
        assert lib.lgh_stage_read_logits(eng._h, again.ctypes.data) == 0
        assert np.array_equal(got.view(np.uint32), again.view(np.uint32)), (vocab, i)
    eng.close()


@pytest.mark.parametrize("vocab,n", [(150, 64), (8191, 64), (12001, 64), (40001, 40)])
def test_rows_apart(pkg, vocab, n):
    parsed = pkg.layered_model.parse_config(lc.config([lc.attn(), lc.mem()], vocab=vocab))
    rng = np.random.default_rng(3)

    class Source:
        def get(self, name, shape):
            v = (rng.standard_normal(shape) / (np.sqrt(shape[-1]) if len(shape) > 1 else 1.0)).astype(np.float32)
            return 30, (v.reshape(-1).view(np.uint32) >> 16).astype(np.uint16)

    eng = pkg.HipGpuInference.from_layered(pkg.LayeredModel(parsed, Source()), n + 8)
    toks = ((np.arange(n) * 37 + 5) % vocab).astype(np.uint32)
    rows = eng.eval(toks, range(n))
    for first, step in ((0, 2), (1, 2), (n - 1, 1)):
        eng.reset()
        want = list(range(first, n, step))
        some = eng.eval(toks, want)
        for i, w in enumerate(want):   # (fewer rows may be another kernel's: bf16 inputs, 2^-8 of the largest)
            assert np.abs(some[i] - rows[w]).max() <= 2.0 ** -8 * np.abs(rows).max(), (vocab, w)
    eng.close()
