"""Build-level properties of the HIP kernels (cross-compiled here, no GPU needed).

A kernel that touches scratch memory pays for the scratch setup at every launch: measured -3.5 % end to end when a
struct was passed to the epilogue by pointer, and again when a per-pass array was indexed by the pass number.  The
compiler reports it; this keeps it at zero for every kernel on the decode path."""
import functools
import os
import re
import subprocess

import __graft_entry__ as graft

CSRC = os.path.join(graft.PKG_DIR, "csrc")
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off", "-mllvm", "-amdgpu-kernarg-preload-count=8",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Rpass-analysis=kernel-resource-usage", "--cuda-device-only", "-c"]


@functools.cache
def _usage(src):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    out = subprocess.run([hipcc, *FLAGS, os.path.join(CSRC, src), "-o", os.devnull], capture_output=True, text=True, check=True).stderr
    res, name = {}, None
    for line in out.splitlines():
        m = re.search(r"Function Name: (\S+)", line)
        if m:
            name = m.group(1)
            res[name] = {}
        m = re.search(r"remark:\s+([A-Za-z ]+?)(?: \[[^\]]*\])?: (\d+)", line)
        if m and name:
            res[name][m.group(1).strip()] = int(m.group(2))
    return res


def test_no_kernel_uses_scratch_or_spills_vgprs():
    for src in ("matvec_mfma.hip", "matvec_batch.hip", "prefill.hip", "attention.hip", "attention_tq.hip", "misc.hip", "dequant.hip",
                "linear_bf16.hip", "latent_attention.hip", "tied_attention.hip", "gated_attention.hip", "moe_route.hip", "mlstm.hip",
                "gla.hip", "glru.hip", "delta.hip", "layered_misc.hip"):
        usage = _usage(src)
        assert usage, f"no kernels found in {src}"
        for fn, u in usage.items():
            assert u.get("ScratchSize", 0) == 0, f"{src}: {fn} uses {u['ScratchSize']} B/lane of scratch"
            assert u.get("VGPRs Spill", 0) == 0, f"{src}: {fn} spills {u['VGPRs Spill']} VGPRs"


def test_mfma_kernel_fits_two_waves_per_simd():
    usage = _usage("matvec_mfma.hip")
    mvq = {fn: u for fn, u in usage.items() if "mvq_kernel" in fn}
    assert len(mvq) == 7   # five formats + the Q4_K/Q6_K and Q5_K/Q6_K mixes
    for fn, u in mvq.items():
        assert u["VGPRs"] <= 256 and u.get("Occupancy", 2) >= 2, (fn, u)


def test_prefill_gemm_keeps_its_accumulators_in_registers():
    """128 f32 accumulators per lane (4 row tiles x 8 token tiles) live in the accumulation registers; one wave per SIMD."""
    usage = _usage("prefill.hip")
    gemm = {fn: u for fn, u in usage.items() if "pf_gemm_kernel" in fn}
    assert len(gemm) == 8   # five formats, the Q4_K/Q6_K and Q5_K/Q6_K mixes, and the any-mix instantiation
    for fn, u in gemm.items():
        assert u.get("AGPRs", 0) >= 128 and u["VGPRs"] <= 256, (fn, u)


def test_long_prompt_kernels_use_no_scratch_and_keep_their_sums_in_registers():
    """prefill_wide.hip: 256 f32 accumulators per lane, one wave per SIMD; attention_wide.hip: two waves per SIMD."""
    for src in ("prefill_wide.hip", "attention_wide.hip"):
        usage = _usage(src)
        assert usage, f"no kernels found in {src}"
        for fn, u in usage.items():
            assert u.get("ScratchSize", 0) == 0 and u.get("VGPRs Spill", 0) == 0, f"{src}: {fn}: {u}"
            if "pw_gemm_kernel" in fn:
                assert u.get("AGPRs", 0) >= 256 and u["VGPRs"] <= 256, (fn, u)
            if "attn_wide_kernel" in fn:
                assert u["VGPRs"] + u.get("AGPRs", 0) <= 256 and u.get("Occupancy", 2) >= 2, (fn, u)


def test_dense_block_products_keep_their_accumulators_in_registers():
    """Dense layers' products of a prompt block (pf_rows_kernel, pf_pair_kernel, pf_pair_few_kernel): 16 f32 accumulators a lane and tile of 32 tokens, two waves a SIMD."""
    usage = _usage("prefill.hip")
    for pattern, count in ((r"pf_rows_kernelILj\d+ELi(\d)E", 8 * 4), (r"pf_pair_kernelILi\d+ELi(\d)E", 5 * 4), (r"pf_pair_few_kernelILi(\d)E", 5)):
        found = {fn: (re.search(pattern, fn), u) for fn, u in usage.items() if re.search(pattern, fn)}
        assert len(found) == count, (pattern, len(found))
        for fn, (m, u) in found.items():
            tiles = 1 if "few" in fn else int(m.group(1))
            assert u["VGPRs"] + u.get("AGPRs", 0) <= 256 and u.get("Occupancy", 2) >= 2, (fn, u)
            assert u["VGPRs"] + u.get("AGPRs", 0) >= 16 * tiles, (fn, u)
