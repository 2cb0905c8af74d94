"""SwiGLU's activation of a mixture's prompt blocks in bf16 (device_utils.h, silu_act_f) where its exponential ends: gates around and far below -88, infinite ones and what is no number, with factors that lift the
smallest results into the logits.  Below -88.8 the activation is -0 in 32 bits, so the logits are those of a model whose gates are zero, bit for bit; above, and for what is no number, the block is held
against the token-by-token path, which takes the library's exponential and division.

Tolerance: bf16 rounding of operands, as in test_gpu_layered."""
import numpy as np
import pytest

import layered_cases as lc

pytestmark = pytest.mark.gpu


def _engine(pkg, gate, up, experts):
    """Channel 8 of the mixture's input is 1 (its norm scales nothing and adds 1), so every gate of the shared feed-forward, and of the experts if they are to have it, is `gate` and every factor `up`."""
    cfg = lc.sandwich([lc.tied(mlp=lc.moe(experts=4, top=1, ff=64, shared=64))], width=128, vocab=300)
    W = lc.clear_calls(lc.Weights(lc.parse(pkg, cfg)), cfg)
    W["l0.norm2"][8], W["l0.norm2.b"][8], W["l0.canon2"][8] = 0.0, 1.0, 0.0
    for part in ("shared", "e0", "e1", "e2", "e3"):
        for name, v in (("gate", gate), ("up", up)):
            W[f"l0.mlp.{part}.{name}"][:] = 0.0
            W[f"l0.mlp.{part}.{name}"][:, 8] = v if part == "shared" or experts else 0.0
    return lc.make(pkg, cfg, "bf16", weights=W)[0]


TOKENS = lc.tokens(40, 300)


@pytest.mark.parametrize("gate", [-400.0, -1e4, -1e30, -3e38])
def test_gates_far_below(pkg, gpu, gate):
    far, none = _engine(pkg, gate, 1e30, True), _engine(pkg, 0.0, 1e30, True)
    got, want = far.eval(TOKENS, range(40)), none.eval(TOKENS, range(40))
    assert np.isfinite(want).all() and np.array_equal(got, want)
    far.close()
    none.close()


@pytest.mark.parametrize("gate,up", [(-88.5, 1e36), (-87.5, 1e36), (-80.0, 1e33), (-20.0, 1e7), (90.0, 0.01), (1e30, 1e-30)])
def test_gates_near_the_end(pkg, gpu, gate, up):
    eng = _engine(pkg, gate, up, False)
    got = eng.eval(TOKENS, range(40))
    eng.reset()
    lc.check(got, lc.stepwise(eng, TOKENS).astype(np.float64), "bf16", f"gate {gate}")
    eng.close()


@pytest.mark.parametrize("gate", [np.inf, -np.inf, np.nan])
def test_gates_that_are_no_number(pkg, gpu, gate):
    eng = _engine(pkg, gate, 0.01, False)
    got = eng.eval(TOKENS, range(40))
    eng.reset()
    assert np.array_equal(np.isnan(got), np.isnan(lc.stepwise(eng, TOKENS)))
    eng.close()
