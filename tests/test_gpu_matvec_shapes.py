"""The single-sequence mat-vec launches (one instantiation per thing done with the rows, the input once per workgroup in LDS) at
the sizes where their geometry changes: fewer slices than waves, slices without blocks, partial workgroups, RoPE rows that do
not fit their place in LDS, two experts' inputs that do not fit side by side.

Tolerances: mat-vecs as the operator tests, 1e-4 sum |x w| + 1e-6 (k / 16 + 20 roundings of 2^-24 of a partial sum that is at most sum |x w|: 1.2e-4 for the largest k if all fell to one side, which they
do not); models as tests/test_gpu_model.py, 2e-3 of the largest logit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TYPES = {"Q4_K": 12, "Q5_K": 13, "Q6_K": 14, "Q8_0": 8, "Q4_0": 2}


@pytest.mark.parametrize("quant", sorted(TYPES))
@pytest.mark.parametrize("k,n", [(256, 16), (512, 40), (768, 33), (1280, 4112), (1792, 48), (2304, 100), (2816, 4096), (5632, 24), (7168, 272), (31744, 16)])
def test_rows_of_every_geometry(pkg, orc, quant, k, n):
    hb, syn = pkg.hip_backend, pkg.synth
    t = TYPES[quant]
    w = syn.fill_tensor("shape.weight", t, k * n, k)
    x = np.random.default_rng(k + n).standard_normal(k).astype(np.float32)
    be = hb.HipBackend()
    got = np.asarray(be.vec_mat_q(x, t, w, n), dtype=np.float64)
    deq = orc.dequantize(t, w, k * n).astype(np.float64).reshape(n, k)
    want, scale = deq @ x.astype(np.float64), np.abs(deq) @ np.abs(x).astype(np.float64)
    assert np.all(np.abs(got - want) <= 1e-4 * scale + 1e-6), (quant, k, n, np.max(np.abs(got - want) / scale))


MODELS = [("test-dense", "Q4_K_M", dict(num_heads=8, num_kv_heads=4, head_dim=288, hidden_size=2304, intermediate_size=2816, num_layers=1)),   # three slices empty; RoPE rows from global memory
          ("test-dense", "Q8_0", dict(num_heads=4, num_kv_heads=4, head_dim=64, hidden_size=256, intermediate_size=512, num_layers=2)),        # one slice, eight row groups
          ("test-dense", "Q5_K_M", dict(num_heads=10, num_kv_heads=2, head_dim=128, hidden_size=1280, intermediate_size=1792, num_layers=2)),  # five slices, seven slices
          ("test-moe", "Q5_K_M", dict(hidden_size=512, num_heads=4, num_kv_heads=2, head_dim=128, intermediate_size=15360, expert_intermediate_size=15360, num_layers=1, num_experts=4, num_experts_per_token=2)),   # the largest two inputs side by side
          ("test-moe", "Q4_K_M", dict(hidden_size=512, num_heads=4, num_kv_heads=2, head_dim=128, intermediate_size=16640, expert_intermediate_size=16640, num_layers=1, num_experts=4, num_experts_per_token=3))]   # one expert a launch


@pytest.mark.parametrize("name,mix,kw", MODELS)
def test_models_of_every_geometry(pkg, orc, name, mix, kw):
    cfg = pkg.make_config(name, max_seq_len=32, **kw)
    model = pkg.SynthModel(cfg, mix=mix)
    ref = orc.Model(cfg.as_dict())
    for nm, t, ne, data in model.tensors(keep=True):
        ref.add_tensor(nm, t, ne, data)
    ref.finalize()
    eng = pkg.HipGpuInference.from_model(model, 32)
    for i in range(6):
        tok = (37 * i + 5) % cfg.vocab_size
        got, want = eng.forward(tok), ref.forward([tok])
        assert np.abs(got - want).max() <= 2e-3 * float(np.abs(want).max()) + 2e-3, (name, kw, i)
    eng.close()
    ref.close()
