"""The grid's strip layout (epirust_amd/csrc/model.hpp), compiled for the host with g++ (the same
functions the kernels use)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_every_neighbourhood_lies_in_one_strip(tmp_path):
    exe = str(tmp_path / "strips_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "epirust_amd", "csrc"),
                           os.path.join(HERE, "native", "strips_check.cpp"), "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout
