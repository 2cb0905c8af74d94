"""Single-sequence mat-vec kernels other than the fused QKV's: what the compiler gives them (no GPU needed)."""
import importlib.util
import os

_spec = importlib.util.spec_from_file_location("test_build_props", os.path.join(os.path.dirname(__file__), "test_build_props.py"))
_props = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(_props)


def test_every_kind_of_rows_fits_two_waves_per_simd():
    found = {fn: u for fn, u in _props._usage("matvec_mfma.hip").items() if "mvq_rows_kernel" in fn}
    assert len(found) == 5 * 4   # formats x (store / residual, SwiGLU, experts' SwiGLU, experts' down)
    for fn, u in found.items():
        assert u["VGPRs"] <= 256 and u.get("Occupancy", 2) >= 2 and u.get("ScratchSize", 0) == 0, (fn, u)
