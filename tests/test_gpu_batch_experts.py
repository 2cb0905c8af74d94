"""gate | up of a mixture's experts in a batched step of few sequences (matvec_batch.hip: mvqb_few_kernel): every format it takes, plans of one to eight k-slices (one with blocks for seven of the eight), a last
workgroup with half its tiles, experts of one entry, two, and more (another turn), and the sequences from which mvqb2 takes over.

Per (row, entry) the kernel does the single-sequence kernel's operations in its order, so the bound is equality of all bits with a single-sequence engine that runs the split attention too (attn_direct=255)."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mix,hidden,kw", [
    ("Q4_K_M", 512, {}), ("Q5_K_M", 1024, {}), ("Q6_K", 2048, {}), ("Q8_0", 512, {}), ("Q8_0", 2048, {}), ("Q4_0", 1024, {}),
    ("Q5_K_M", 3328, dict(expert_intermediate_size=10496)), ("Q4_K_M", 4096, {}),
    ("Q6_K", 1024, dict(num_experts=8, num_experts_per_token=1)), ("Q4_K_M", 2048, dict(num_experts=12, num_experts_per_token=4)),
])
def test_experts_of_few_entries_are_bitwise_the_single_sequence(pkg, mix, hidden, kw):
    over = dict(hidden_size=hidden, num_heads=hidden // 64, num_kv_heads=hidden // 128, num_layers=1, num_experts=8, expert_intermediate_size=10240)
    over.update(kw)
    cfg = pkg.make_config("test-moe", max_seq_len=32, **over)
    model = pkg.SynthModel(cfg, mix=mix)
    multi = pkg.HipGpuInference.from_model(model, 32)
    single = pkg.HipGpuInference.from_model(model, 32, attn_direct=255)
    multi.batch_create(12)
    tok = np.random.default_rng(7).integers(0, cfg.vocab_size, (12, 2))
    tok[5:9] = tok[5]                                  # four sequences alike: their experts have four entries
    want = []
    for s in range(12):
        single.reset()
        want.append([single.forward(int(t)).copy() for t in tok[s]])
    for n in (2, 3, 5, 8, 12):
        for s in range(12):
            multi.batch_reset(s)
        for step in range(2):
            got, _ = multi.forward_multi(list(range(n)), tok[:n, step])
            for s in range(n):
                assert np.array_equal(got[s].view(np.uint32), want[s][step].view(np.uint32)), (n, s, step)
    multi.close()
    single.close()


@pytest.mark.parametrize("mix,hidden,ff,slots", [("Q4_K_M", 2048, 2048, 2), ("Q8_0", 2048, 5632, 3), ("Q5_K_M", 2048, 5632, 7)])
def test_experts_in_eight_slices_have_room_for_their_sums(pkg, mix, hidden, ff, slots):
    """Experts whose gate | up is split into eight k-slices, and wider than half the hidden size: their partial sums are the most that a step holds (lgh_batch_create sizes the buffer, and launches its steps)."""
    cfg = pkg.make_config("test-moe", max_seq_len=32, hidden_size=hidden, num_heads=hidden // 64, num_kv_heads=hidden // 128, num_layers=1, num_experts=8, expert_intermediate_size=ff)
    multi = pkg.HipGpuInference.from_model(pkg.SynthModel(cfg, mix=mix), 32)
    multi.batch_create(slots)
    tok = np.random.default_rng(11).integers(0, cfg.vocab_size, (slots, 2))
    got = [multi.forward_multi(list(range(slots)), tok[:, step])[0].copy() for step in range(2)]
    for s in range(slots):
        multi.reset()
        for step in range(2):
            want = multi.forward(int(tok[s, step]))
            assert np.array_equal(got[step][s].view(np.uint32), want.view(np.uint32)), (s, step)
    multi.close()


_FRESH = """
import sys
sys.path.insert(0, sys.argv[1])
import numpy as np
import __graft_entry__ as graft
pkg = graft.load_package()
cfg = pkg.make_config("test-moe", max_seq_len=32, num_layers=1, num_experts=int(sys.argv[3]), expert_intermediate_size=int(sys.argv[6]))
multi = pkg.HipGpuInference.from_model(pkg.SynthModel(cfg, mix=sys.argv[2]), 32)
slots, n = int(sys.argv[4]), int(sys.argv[5])
multi.batch_create(slots)
tok = np.random.default_rng(7).integers(0, cfg.vocab_size, (n, 4))
got = [multi.forward_multi(list(range(n)), tok[:, i])[0].copy() for i in range(4)]
for s in range(n):
    multi.reset()
    for i in range(4):
        want = multi.forward(int(tok[s, i]))
        assert np.array_equal(got[i][s].view(np.uint32), want.view(np.uint32)), (s, i)
print("equal")
"""


def _in_fresh_process(mix, experts, slots, n, ff, **env):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", _FRESH, root, mix, str(experts), str(slots), str(n), str(ff)], capture_output=True, text=True, timeout=100, env=dict(os.environ, **env))
    assert out.returncode == 0 and out.stdout.strip().endswith("equal"), out.stdout + out.stderr


@pytest.mark.parametrize("mix,experts,slots,n", [("Q8_0", 8, 8, 7), ("Q5_K_M", 5, 7, 7)])
def test_first_step_of_a_size_in_a_fresh_process(mix, experts, slots, n):
    """A kernel whose first launch in the process happens during a capture is not replayed with the graph: the sizes from which mvqb2 takes over lie inside its groups of up to 4, 8 and 16, so lgh_batch_create launches
    the largest of each group as well."""
    _in_fresh_process(mix, experts, slots, n, 10240)


@pytest.mark.parametrize("least,slots,n", [(3, 2, 2), (5, 4, 4)])
def test_fewer_sequences_than_the_kernels_with_entry_lists_take(least, slots, n):
    """LGH_MVQB2_MIN keeps smaller steps from the kernels that take entry lists: a mixture's sequences go one after the other there."""
    _in_fresh_process("Q5_K_M", 4, slots, n, 1024, LGH_MVQB2_MIN=str(least))
