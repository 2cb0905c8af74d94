"""The residual stream behind the first layer of a prompt block, every token of it, beside the exact token-by-token path's (a stage of one layer keeps both)."""
import ctypes

import numpy as np


def check(pkg, model, sizes):
    """A layer's five products and its attention follow each other, each with operands rounded to 11 bits: 2^-10 of their own norm at most, together below 6e-3 of a token's; a tile of 16 rows that misses 256 of its
    columns is off by more than 2e-2 in some token."""
    cfg = model.config
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    block, exact = (pkg.HipGpuInference.from_model(model, 160, layer_range=(0, 1)) for _ in range(2))
    assert block.prefill_is_batched()
    for n in sizes:
        prompt = [(11 * i + n) % cfg.vocab_size for i in range(n)]
        block.reset()
        exact.reset()
        block.stage_prefill_batch(prompt, n)
        block.synchronize()
        got, want = np.empty((n, cfg.hidden_size), np.float32), np.empty((n, cfg.hidden_size), np.float32)
        assert hip.hipMemcpy(got.ctypes.data, block.stage_hidden_block_ptr(), got.nbytes, 2) == 0   # to the host
        for i, t in enumerate(prompt):
            exact.stage_forward(t)
            want[i] = exact.read_hidden()
        off = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
        assert np.isfinite(got).all() and off.max() <= 1e-2, (n, int(off.argmax()), float(off.max()))
    block.close()
    exact.close()
