"""The 16-bit steps of two cells per thread, compiled for the host: a cell that
stores nothing keeps what another writer (a face transfer on another stream) puts
into its slots while its neighbour in the pair is stepped, for every pair of
flags, both half-steps and the three formats; the neighbour's bits are those of
the one-cell code. Only the OBSTACLE cells of a closed domain may be stored back."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
CLANG = shutil.which("amdclang++") or os.path.join(ROCM, "llvm", "bin", "clang++")


@pytest.mark.skipif(not os.path.exists(CLANG), reason="needs the ROCm clang")
def test_still_cell_of_a_pair_is_not_stored(tmp_path):
    exe = str(tmp_path / "step_pairs")
    subprocess.run([CLANG, "-x", "c++", "-std=c++17", "-O1", "-ffp-contract=off", "-w",
                    "-I", os.path.join(ROCM, "include"), "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "cavityflow_cuda_amd", "csrc"),
                    os.path.join(ROOT, "tests", "step_pairs_host.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout
    assert out.stdout.strip() == "%d cases" % (2 * 3 * 2 * 4 * 4)
