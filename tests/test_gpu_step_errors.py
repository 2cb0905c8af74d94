"""A step that fails, or that finds an error which is not its own: the device's position word and the host's count stay together (engine.hip: step).  A context that had the trouble has, call by call, the bits and the
position of one that had none."""
import ctypes
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ROWS = 12


@pytest.fixture(scope="module")
def pair(pkg):
    made = []

    def make(flags=0, mix="Q4_K_M", **kw):
        cfg = pkg.make_config("test-dense", max_seq_len=ROWS)
        model = pkg.SynthModel(cfg, mix=mix)
        made.extend(pkg.HipGpuInference.from_model(model, ROWS, flags=flags, **kw) for _ in range(2))
        return made[-2:]

    yield make
    for e in made:
        e.close()


def leave_an_error(pkg):
    """An ordinary refused call of the program's: no such device."""
    lib = re.search(r"\S*libamdhip64\S*", open("/proc/self/maps").read()).group(0)   # the runtime that the engine uses
    hip = ctypes.CDLL(lib)
    assert hip.hipSetDevice(pkg.hip_backend.device_count() + 7) != 0
    return hip.hipPeekAtLastError()


def same(a, b):
    return np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("flags", [0, 1], ids=["graph", "no-graph"])
def test_an_error_left_by_another_library(pkg, pair, flags):
    a, b = pair(flags)
    b.forward(900)
    assert leave_an_error(pkg) != 0          # it is there, and for a step's launches to find
    b.reset()
    for i in range(ROWS):                    # up to the last row
        leave_an_error(pkg)
        if i % 3 == 1:
            a.prefill_token(5 * i + 1)
            b.prefill_token(5 * i + 1)
        elif i % 3 == 2:
            assert a.forward_argmax(5 * i + 1) == b.forward_argmax(5 * i + 1)
        else:
            assert same(a.forward(5 * i + 1), b.forward(5 * i + 1)), i
        assert a.position() == b.position() == i + 1
    with pytest.raises(pkg.BackendError):
        b.forward(1)


# in a graph's step the first launch is the embedding's, outside of the graph, the second the graph; without one every kernel is a launch: the first ones, some in a layer
@pytest.mark.parametrize("flags,nth", [(0, 1), (0, 2), (1, 1), (1, 2), (1, 5), (1, 9)])
def test_a_step_that_fails_is_as_if_it_had_not_been(pkg, pair, flags, nth):
    a, b = pair(flags)
    for i in range(ROWS):                    # the last row among them: a position that had run ahead would be behind the cache there
        tok = 7 * i + 3
        if i:                                # (graphs are captured at the first token)
            for call in (b.forward, b.prefill_token):
                b.debug_fail_launch(nth)
                with pytest.raises(pkg.BackendError):
                    call(tok)
                b.debug_fail_launch(0)
                assert b.position() == i
        if i == 0:
            a.prefill_token(2), b.prefill_token(2)
            a.reset(), b.reset()
        assert same(a.forward(tok), b.forward(tok)), i
        assert same(a.read_hidden(), b.read_hidden()), i


def test_greedy_steps_that_fail(pkg, pair):
    a, b = pair()
    want = a.decode_greedy(11, ROWS)
    b.decode_greedy(11, 2)
    b.reset()
    b.debug_fail_launch(4)                   # the fourth token's graph
    with pytest.raises(pkg.BackendError):
        b.decode_greedy(11, ROWS)
    b.debug_fail_launch(0)
    assert b.position() == 3
    assert np.array_equal(b.decode_greedy(int(want[2]), ROWS - 3), want[3:])


def test_eval_behind_a_failed_step(pkg, pair):
    a, b = pair()
    prompt = [3, 1, 4, 1, 5, 9]
    for e in (a, b):
        e.forward(1), e.reset()
    b.debug_fail_launch(1)
    with pytest.raises(pkg.BackendError):
        b.forward(8)
    b.debug_fail_launch(0)
    for e in (a, b):
        e.forward_batch(prompt)
    for tok in (2, 6, 5):
        assert same(a.forward(tok), b.forward(tok))
