"""Block products of layer-by-layer models whose tiles give every CU one at most (linear_bf16.hip, two teams of waves a workgroup): tiles of 64, 96 and 128 tokens with whole and ragged ends, inner sizes
of whole k-steps and with a remainder.  Vocabularies of 118 and 235 weight panels bring the head there at these token counts.  Against the oracle, to bf16 rounding of operands as in test_gpu_layered."""
import pytest

import layered_cases as lc
from oracle import layered as lo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,vocab,tokens", [
    (1024, 15001, (65, 100, 128)),                # two tiles of 64
    (1090, 30000, (33, 64, 65, 96, 97, 128)),     # one of 64, of 96, of 128
    (1024, 30003, (40, 80, 120)),
])
def test_one_tile_a_cu(pkg, gpu, width, vocab, tokens):
    cfg = lc.config([lc.mem(ff=50)], width=width, vocab=vocab)
    eng, W = lc.make(pkg, cfg, "bf16", max_seq=160)
    toks = lc.tokens(128, cfg["vocab"])
    want = lo.forward(cfg, W, toks)
    for n in tokens:
        eng.reset()
        lc.check(eng.eval(toks[:n], range(n)), want[:n], "bf16", f"{n} tokens")
    eng.close()


def test_tiles_of_160(pkg, gpu):
    """Where two workgroups a CU would take two rounds of tiles of 128 and take one of 160: the joint input product (32 896 columns, 257 panels) and the gated feed-forward's first (33 200 columns,
    260 panels); whole and ragged ends, and one token beyond a tile."""
    cfg = lc.config([lc.mem(heads=64, dim=128, vdim=128, ff=16600)], width=1024, vocab=300)
    eng, W = lc.make(pkg, cfg, "bf16", max_seq=200)
    toks = lc.tokens(161, cfg["vocab"])
    want = lo.forward(cfg, W, toks)
    for n in (129, 145, 160, 161):
        eng.reset()
        lc.check(eng.eval(toks[:n], range(n)), want[:n], "bf16", f"{n} tokens")
    eng.close()
