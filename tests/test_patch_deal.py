"""How input patches of the fused inverted residual block are dealt to threads."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_every_unit_is_dealt_once_and_patches_of_many_blocks_are_fetched_ahead(tmp_path):
    exe = str(tmp_path / "patch_deal_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", os.path.join(HERE, "patch_deal_check.cpp"), "-o", exe])
    assert subprocess.run([exe], capture_output=True, text=True).stdout.strip() == "ok"
