"""Requantisation by table address computes with f32 denormals: the build's flags keep them, whatever the compiler's default is."""
import os
import re
import subprocess
import sys

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "z-ant_amd")


def test_kernels_are_built_with_f32_denormals(tmp_path, monkeypatch):
    monkeypatch.syspath_prepend(PKG)
    monkeypatch.delitem(sys.modules, "build", raising=False)
    import build
    assert "-fno-gpu-flush-denormals-to-zero" in build.FLAGS
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text('#include "qblock_i8.h"\n'
                   "__global__ void probe(unsigned *y, const int *x, float m, RequantLut t) { y[threadIdx.x] = requant_entry(x[threadIdx.x], m, t); }\n")
    # a flag in front that asks for the opposite stands for a compiler that flushes by default
    subprocess.check_call([build.HIPCC, "-fgpu-flush-denormals-to-zero"] + build.FLAGS + ["-S", "--cuda-device-only", str(src), "-o", str(out)],
                          stderr=subprocess.DEVNULL)
    assert re.findall(r"float_denorm_mode_32 (\d)", out.read_text()) == ["3"]
    monkeypatch.delitem(sys.modules, "build", raising=False)
