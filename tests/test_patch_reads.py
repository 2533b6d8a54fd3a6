"""The bank-conflict model that chooses the int8 convolution's patch pitch, against its definition lane by lane."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_patch_reads_agree_with_the_definition(tmp_path):
    exe = str(tmp_path / "patch_reads_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", os.path.join(HERE, "patch_reads_check.cpp"), "-o", exe])
    assert subprocess.check_output([exe], text=True).strip() == "ok"
