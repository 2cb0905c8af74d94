"""The rules by which calls choose their kernels (csrc/dispatch_rules.h), compiled for the host."""
import os
import subprocess

import __graft_entry__ as graft


def test_rules_on_the_host(tmp_path):
    exe = str(tmp_path / "dispatch_rules_test")
    here = os.path.dirname(os.path.abspath(__file__))
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(graft.PKG_DIR, "csrc"), os.path.join(here, "cpp", "dispatch_rules_test.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
