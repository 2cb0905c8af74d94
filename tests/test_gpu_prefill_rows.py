"""Products of a prompt block of up to 128 tokens (prefill.hip, pf_rows_kernel) against the dequantized product in 64 bits: token counts around the tiles of 32, one to seven blocks of 256 columns in a k-range
(the loop takes three a turn, one or two are left over), rows that leave half a unit of 32 or a workgroup of 128 unfilled, every format.

Tolerance: operands rounded to 11 significant bits each, sums in f32: |d| <= 2^-10 * sum |x w| covers both roundings (2^-11 each) with the sums' rounding far below."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tname", ["Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q4_0"])
@pytest.mark.parametrize("k,n,tokens", [
    (256, 16, (1, 32, 33)),          # one block: the loop has no turn; half a unit
    (512, 48, (31, 64, 65)),         # a tile and a half of 32 rows
    (768, 16384, (96, 128)),         # 128 workgroups of two k-ranges, of two blocks and of one
    (2048, 16384, (97, 127)),        # four blocks a range: a turn and one
    (1280, 4112, (50, 80)),          # 33 workgroups, the last with one tile
    (7168, 8192, (16, 128)),         # seven blocks a range: two turns and one
])
def test_block_product_matches_dequantized(gpu, pkg, orc, tname, k, n, tokens):
    t = pkg.synth.TYPE_IDS[tname]
    raw = pkg.synth.fill_tensor("blk.0.test.weight", t, k * n, k)
    w = orc.dequantize(t, raw, k * n).reshape(n, k)
    pick = np.unique(np.concatenate([np.arange(min(n, 160)), np.arange(max(0, n - 160), n)]))
    w64 = w[pick].astype(np.float64)
    for m in tokens:
        x = np.random.default_rng(k + n + m).standard_normal((m, k)).astype(np.float32)
        got = gpu.op_mat_mat(t, raw, x, n)
        x64 = x.astype(np.float64)
        bound = 2.0 ** -10 * (np.abs(x64) @ np.abs(w64).T) + 1e-6
        assert np.isfinite(got).all() and (np.abs(got[:, pick] - x64 @ w64.T) <= bound).all(), m
