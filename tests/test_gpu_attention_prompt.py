"""The attention of long prompt blocks (attention_wide.hip) by itself, its sums in f32, against the same in 64 bits.

Bound per value, from f32 arithmetic alone: a score is a sum of D products, off by at most (D + 4) * 2^-24 of sum |q k| (the product and its sums; the scale, the
limbs that are left out); a weight is off by what its score and the largest one are off and 8 * 2^-24 for the exponential and the merge of two maxima;
the weighted sum adds (rows + 4) * 2^-24 of sum w |v|.  It holds whatever the other rows and tokens hold.
In earnest roundings cancel: ordinary inputs are off by 1e-7 to 5e-7 (2-norm); 1e-6 is demanded."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


def _run(pkg, q, kc, vc, pos0):
    m, heads, d = q.shape
    out = np.empty_like(q)
    rc = pkg.hip_backend.load_library().lgh_op_attention_prompt(0, q.ctypes.data, kc.ctypes.data, vc.ctypes.data, out.ctypes.data, heads, kc.shape[0], d, kc.shape[1],
                                                                C.c_float(d ** -0.5), pos0, m)
    assert rc == 0, rc
    return out


def _check(q, kc, vc, pos0, out, ordinary=False):
    m, heads, d = q.shape
    n_kv, rows = kc.shape[0], pos0 + m
    scale = float(np.float32(d ** -0.5))
    off, norm = 0.0, 0.0
    for h in range(heads):
        Q = torch.from_numpy(q[:, h]).double()
        K, V = (torch.from_numpy(x[h // (heads // n_kv), :rows]).double() for x in (kc, vc))
        hide = torch.arange(rows)[None, :] > pos0 + torch.arange(m)[:, None]
        s = (Q @ K.T * scale).masked_fill(hide, -torch.inf)
        w = torch.softmax(s, -1)
        ds = (d + 4) * U * scale * (Q.abs() @ K.abs().T)
        top = ds.gather(1, s.argmax(-1, keepdim=True))
        want, mass = w @ V, w @ V.abs()
        dw = torch.expm1(ds + top + 8 * U).clamp(max=1e30)
        bound = (w * dw) @ V.abs() + mass * (w * dw).sum(-1, keepdim=True) + (rows + 4) * U * mass
        got = torch.from_numpy(out[:, h]).double()
        over = (got - want).abs() - bound
        assert bool((over <= 0).all()), (h, float(over.max()), [int(i) for i in np.unravel_index(int(over.argmax()), over.shape)])
        off += float((got - want).square().sum())
        norm += float(want.square().sum())
    if ordinary:
        assert (off / norm) ** 0.5 <= 1e-6, (off / norm) ** 0.5
    return (off / norm) ** 0.5


def _inputs(d, heads, n_kv, pos0, m, seed):
    rng = np.random.default_rng(seed)
    q, kc, vc = (rng.standard_normal(s, dtype=np.float32) for s in ((m, heads, d), (n_kv, pos0 + m + 3, d), (n_kv, pos0 + m + 3, d)))
    kc[:, pos0 + m:], vc[:, pos0 + m:] = np.nan, np.nan      # rows past the block: never used
    return q * 2.0, kc, vc


@pytest.mark.parametrize("d,heads,n_kv,pos0,m", [
    (64, 4, 4, 0, 1), (64, 8, 1, 0, 31), (128, 4, 2, 0, 33), (128, 8, 2, 5, 127), (128, 4, 4, 31, 128), (64, 8, 4, 33, 129), (128, 8, 1, 64, 257),
    (64, 16, 2, 700, 300), (128, 16, 4, 0, 511), (128, 3, 3, 1, 1025),
    (64, 40, 40, 0, 2047),                                    # more than two workgroups a CU
    (128, 4, 1, 1100, 40), (64, 8, 8, 9000, 70), (128, 8, 1, 3001, 129), (64, 8, 2, 1050, 511)])   # few tokens behind many rows: splits, 2 to 16 of them
def test_ordinary_inputs(pkg, d, heads, n_kv, pos0, m):
    q, kc, vc = _inputs(d, heads, n_kv, pos0, m, 7 * m + d)
    print("relative error", _check(q, kc, vc, pos0, _run(pkg, q, kc, vc, pos0), ordinary=True))


@pytest.mark.parametrize("d,heads,n_kv", [(128, 4, 1), (64, 2, 2)])
@pytest.mark.parametrize("what", ["a large key", "a large value that is not looked at", "small values", "channels of a key", "a later value"])
def test_rows_of_very_different_size(pkg, d, heads, n_kv, what):
    """What a row holds decides its own part alone, however far its neighbours lie from it."""
    pos0, m = 3, 200
    q, kc, vc = _inputs(d, heads, n_kv, pos0, m, 11)
    q[..., 0] = np.abs(q[..., 0]) + 0.5
    if what == "a large key":                                 # far below in every score: the rows beside it share all weights
        kc[:, 37] = 0.0
        kc[:, 37, 0] = -2.0 ** 34
    if what == "a large value that is not looked at":
        kc[:, 37, 0] = -2.0 ** 12
        vc[:, 37] *= 2.0 ** 34
    if what == "small values":                                # the first tile is looked at alone and lies far below the others
        kc[:, 30:, 0] = -2.0 ** 12
        vc[:, :30] *= 2.0 ** -34
    if what == "channels of a key":                           # one channel far above the others, where no query looks
        kc[..., 5] = 2.0 ** 30
        q[..., 5] = 0.0
    if what == "a later value":                               # of the same tile, invisible to the tokens before it
        vc[:, 100] *= 2.0 ** 34
    print("relative error", _check(q, kc, vc, pos0, _run(pkg, q, kc, vc, pos0)))
