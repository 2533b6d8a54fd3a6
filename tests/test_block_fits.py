"""Fused inverted residual blocks and chains of them are taken up to what LDS holds: the tables beside the weights are kept small."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "z-ant_amd")


def test_blocks_and_chains_that_fit_are_taken(tmp_path):
    exe = str(tmp_path / "block_fit_check")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(PKG, "csrc"), "-I", os.path.join(ROOT, "include"),
                           "-I", "/opt/rocm/include", os.path.join(ROOT, "tests", "block_fit_check.cpp"), "-o", exe, "-L", PKG, "-lzant_hip",
                           "-Wl,-rpath," + PKG, "-L", "/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib"])
    assert subprocess.run([exe], capture_output=True, text=True).stdout.strip() == "ok"
