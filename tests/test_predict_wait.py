"""predict on host buffers waits for its upload on every way out."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "z-ant_amd")


def test_the_input_buffer_is_given_back_after_its_upload(tmp_path):
    exe = str(tmp_path / "predict_wait_check")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(PKG, "csrc"), "-I",
                           os.path.join(ROOT, "include"), "-I", "/opt/rocm/include", os.path.join(ROOT, "tests", "predict_wait_check.cpp"), "-o", exe,
                           "-L", PKG, "-lzant_hip", "-Wl,-rpath," + PKG, "-L", "/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib"])
    assert subprocess.run([exe], capture_output=True, text=True).stdout.strip() == "ok"
