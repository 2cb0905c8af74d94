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


def test_every_kernel_belongs_to_one_reported_symbol(pkg):
    """What lgh_get_stats counts launches under, against the kernels that are built: all of them, each in one symbol, no symbol without one."""
    import re
    import subprocess
    names = subprocess.run(["c++filt"], input="\n".join(_props._usage("matvec_mfma.hip")), capture_output=True, text=True, check=True).stdout.splitlines()
    kernels = {re.sub(r"^void |\(.*$", "", n) for n in names if re.search(r"\bmvq_(rows_)?kernel<", n)}
    assert len(kernels) == 7 + 5 * 4
    hb = pkg.hip_backend
    symbols = [s for s in hb.SYM_NAMES if "mvq_" in s]
    found = {s: hb.symbol_rows(s, sorted(kernels)) for s in symbols}
    assert len(symbols) == 5 and all(found.values())
    assert sorted(k for f in found.values() for k in f) == sorted(kernels)


def test_traffic_of_a_symbol_is_that_of_its_kernels(tmp_path):
    """bench.py's bytes a launch: the mean over the kernels of a symbol, and none from a table that lacks one of them (another tree's)."""
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    sys.path.insert(0, root)
    import bench
    head = "kernel,launches_fetch_pass,FETCH_SIZE_KB_mean_raw,launches_write_pass,WRITE_SIZE_KB_mean_raw,hbm_bytes_per_launch_corrected\n"
    old, new = tmp_path / "a_pmc_traffic.csv", tmp_path / "b_pmc_traffic.csv"
    old.write_text(head + "lgh::mvq_kernel<1u>,5856,1,5856,1,33684912\nlgh::mvq_kernel<3u>,976,1,976,1,15912018\n")
    new.write_text(head + 'lgh::mvq_kernel<1u>,10,1,10,1,1000\n"lgh::mvq_rows_kernel<1u, 0>",20,1,20,1,4000\n"lgh::mvq_rows_kernel<1u, 1>",10,1,10,1,7000\n"lgh::mvq_rows_kernel<2u, 1>",10,1,10,1,9\n')
    symbol = "lgh::mvq_kernel<1u> + lgh::mvq_rows_kernel<1u, *>"
    assert bench.committed_traffic(symbol, [old]) == (None, None)
    assert bench.committed_traffic(symbol, [old, new]) == (4000, new.name)
    assert bench.committed_traffic("lgh::mvq_kernel<3u>", [old, new]) == (15912018, old.name)
    assert bench.committed_traffic("lgh::tied_*", [old, new]) == (None, None)
