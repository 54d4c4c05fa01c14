"""The host runtime's decisions (epirust_amd/csrc/engine.cpp) on a device played on the host
(tests/native/fake_device.hpp), compiled with g++."""
import os
import subprocess

import pytest

from epirust_amd import build as B

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def checks(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("engine") / "engine_check")
    sources = [os.path.join(B.SRC, s) for s in ("engine.cpp", "config.cpp", "population.cpp")]
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I" + B.SRC, "-I" + os.path.join(ROOT, "include")] + B.HOST +
                          [os.path.join(HERE, "native", "engine_check.cpp")] + sources + ["-o", exe, "-lpthread"])
    return exe


@pytest.mark.parametrize("check", ["block_size_failure", "rest_hours", "days_after_the_stop",
                                   "graphs_under_a_lockdown", "small_handles_with_an_office_layout"])
def test_engine(checks, check):
    out = subprocess.run([checks, check], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
