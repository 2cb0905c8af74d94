"""Memory of results that are gone serves later ones (hip_backend.ResultMemory): never while a view of the old one is there, never more than the bound."""
import importlib
import threading

import numpy as np
import pytest

ResultMemory = importlib.import_module("llama-gguf_amd.hip_backend").ResultMemory


@pytest.mark.parametrize("shape", [(1,), (7,), (3, 5), (16, 32000)])
def test_a_result_is_its_own_until_the_last_view_is_gone(shape):
    mem = ResultMemory()
    a = mem.take(*shape)
    assert a.shape == shape and a.dtype == np.float32 and a.flags.c_contiguous and a.flags.writeable and mem.idle == 0
    a[...] = 1.0
    view, where = a.reshape(-1)[-1:], a.ctypes.data
    del a
    b = mem.take(*shape)                       # the view keeps the first one's memory
    b[...] = 2.0
    assert view[0] == 1.0 and b.ctypes.data != where and mem.idle == 0
    del view
    assert mem.idle == b.nbytes
    c = mem.take(*shape)
    assert c.ctypes.data == where and mem.idle == 0 and (b == 2.0).all()


def test_no_rows_and_the_bound():
    mem = ResultMemory(limit=4096)
    assert mem.take(0, 8).shape == (0, 8) and mem.idle == 0
    held = [mem.take(256) for _ in range(9)]   # 1 KB each: four stay
    del held
    assert mem.idle == 4096
    big = mem.take(2048)
    del big                                    # more than the bound: not kept
    assert mem.idle == 4096
    other = mem.take(512)
    del other                                  # two of the size that came first make room
    assert mem.idle == 4096 and mem.take(512) is not None and mem.idle == 2048


def test_several_threads_never_share_a_result():
    mem, bad = ResultMemory(limit=1 << 16), []

    def work(k):
        kept = []
        for i in range(400):
            a = mem.take(64 + i % 3)
            a[...] = k * 1000 + i
            kept.append((k * 1000 + i, a))
            if len(kept) > 5:
                want, old = kept.pop(0)
                if not (old == want).all():
                    bad.append((k, i))
    threads = [threading.Thread(target=work, args=(k,)) for k in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad and 0 <= mem.idle <= 1 << 16
