"""The batch autotuner's search, compiled for the host and run on made-up times: the
schedule of a batch without a set tuning is one of its finalists and is chosen where
nothing is faster, from every starting tuning."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
CXX = shutil.which("g++")


@pytest.mark.skipif(not CXX, reason="needs g++")
def test_search_chooses_the_fastest_schedule(tmp_path):
    exe = str(tmp_path / "tuner")
    subprocess.run([CXX, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(ROCM, "include"), "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "cavityflow_cuda_amd", "csrc"),
                    os.path.join(ROOT, "tests", "tuner_host.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout
