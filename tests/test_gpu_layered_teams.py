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


@pytest.mark.parametrize("heads,ff,tokens", [
    (64, 16600, (129, 145, 160)),          # 257 and 260 panels, two tiles of 128 and one of 160
    (50, 12800, (257, 289, 301, 319, 320)),   # 201 and 200 panels, three of 128 and two of 160
])
def test_tiles_of_160(pkg, gpu, heads, ff, tokens):
    """Where two workgroups a CU would take two rounds of tiles of 128 and take one of 160: the joint input product (4 x 128 columns a head and the gates) and the gated feed-forward's first (two columns a unit);
    whole and ragged last tiles, alone and behind a full one."""
    cfg = lc.config([lc.mem(heads=heads, dim=128, vdim=128, ff=ff)], width=1024, vocab=300)
    eng, W = lc.make(pkg, cfg, "bf16", max_seq=360)
    toks = lc.tokens(tokens[-1], cfg["vocab"])
    want = lo.forward(cfg, W, toks)
    for n in tokens:
        eng.reset()
        lc.check(eng.eval(toks[:n], range(n)), want[:n], "bf16", f"{n} tokens")
    eng.close()
