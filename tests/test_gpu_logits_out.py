"""Results on their way to the caller (engine.hip, floats_to_host): pieces of 131 072 floats through a ring of four in pinned memory.  Vocabularies around one piece, and steps of several sequences whose
logits take more pieces than the ring has; every sequence's logits against the same sequence's alone, bit for bit.  Memory of the caller that the device reaches itself gets the same."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab,sequences", [(131072, 2), (131073, 2), (98304, 7), (16385, 16), (48000, 16)])
def test_logits_of_many_pieces(pkg, vocab, sequences):
    cfg = pkg.make_config("test-dense", max_seq_len=16, vocab_size=vocab)
    eng = pkg.HipGpuInference.from_model(pkg.SynthModel(cfg, mix="Q4_K_M"), 16)
    alone = []
    for s in range(sequences):
        eng.reset()
        alone.append([eng.forward((31 * s + k) % vocab) for k in range(2)])
    eng.batch_create(sequences)
    for k in range(2):
        got, _ = eng.forward_multi(list(range(sequences)), [(31 * s + k) % vocab for s in range(sequences)])
        for s in range(sequences):
            assert np.abs(got[s] - alone[s][k]).max() <= 1e-4 * np.abs(alone[s][k]).max(), (s, k)   # (a context without slots may take another order of sums in attention)
            eng.reset()
            want = [eng.forward((31 * s + j) % vocab) for j in range(k + 1)][-1]
            assert np.array_equal(got[s].view(np.uint32), want.view(np.uint32)), (s, k)
    eng.close()


def test_logits_into_pinned_memory(pkg):
    cfg = pkg.make_config("test-dense", max_seq_len=16)
    eng = pkg.HipGpuInference.from_model(pkg.SynthModel(cfg, mix="Q4_K_M"), 16)
    want = eng.forward(7)
    eng.reset()
    lib, p = pkg.hip_backend.load_library(), C.c_void_p()
    hip = C.CDLL(lib._name)   # (the same library: its runtime's functions are found through it)
    assert hip.hipHostMalloc(C.byref(p), C.c_size_t(cfg.vocab_size * 4), C.c_uint(0)) == 0
    assert lib.lgh_forward(eng._h, 7, p) == 0
    out = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_uint32)), (cfg.vocab_size,)).copy()
    assert hip.hipHostFree(p) == 0
    assert np.array_equal(out, want.view(np.uint32))
    eng.close()


def test_the_callers_pages_keep_what_they_hold_until_the_result(pkg):
    """Pages are touched while the device still works: another thread sees in a page's first byte what it held or what the result puts there, nothing else."""
    cfg = pkg.make_config("test-dense", max_seq_len=40, vocab_size=48000)
    eng = pkg.HipGpuInference.from_model(pkg.SynthModel(cfg, mix="Q4_K_M"), 40)
    eng.batch_create(16)
    lib, n = pkg.hip_backend.load_library(), 16
    slots = np.arange(n, dtype=np.uint32)
    buf = np.empty(n * cfg.vocab_size * 4, np.uint8)
    heads, looks = buf[::4096], 0
    for step in range(20):
        tokens = (slots * 31 + step).astype(np.uint32)
        buf[:] = 0xA5
        rc, seen = [], []
        t = threading.Thread(target=lambda: rc.append(lib.lgh_forward_multi(eng._h, slots.ctypes.data, tokens.ctypes.data, n, buf.ctypes.data, None)))
        t.start()
        while t.is_alive():
            seen.append(heads.copy())
        t.join()
        assert rc == [0]
        looks += len(seen)
        odd = [int(((s != 0xA5) & (s != heads)).sum()) for s in seen]
        assert not any(odd), (step, odd)
    assert looks > 0
    eng.close()
