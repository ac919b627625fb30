"""The launch options that whole-domain steps choose, compiled for the host."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
CLANG = shutil.which("amdclang++") or os.path.join(ROCM, "llvm", "bin", "clang++")
pytestmark = pytest.mark.skipif(not os.path.exists(CLANG), reason="needs the ROCm clang")

NT, X, W4, W3, W2, LDS, BIG, PAIR, REV = 1, 2, 4, 8, 16, 128, 256, 1 << 16, 1 << 17
PRECISIONS = {"f32": 0, "f64": 1, "f16s": 2, "bf16s": 3, "f16c": 4}
WALL, GHOST = 1, 8
P = PAIR

# precision, interior size, outputs, one face, MiB of others between (near, far), alpha,
# beta; a last 1: the half-step before was nontemporal
ROWS = [
    # within the L2s, every slab alike
    ("f32", (37, 33, 31), 0, WALL, 0, 0, X, X), ("f32", (62, 62, 62), 0, WALL, 0, 0, X, X),
    ("f32", (62, 62, 62), 1, WALL, 500, 500, X, X), ("f64", (59, 59, 59), 0, WALL, 0, 0, X, X),
    ("f16s", (75, 74, 73), 1, WALL, 0, 0, X, X), ("f16c", (91, 87, 83), 0, GHOST, 0, 0, X, X),
]


def test_chosen_options(tmp_path):
    exe = str(tmp_path / "step_options")
    subprocess.run([CLANG, "-x", "c++", "-std=c++17", "-O1", "-w",
                    "-I", os.path.join(ROCM, "include"), "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "cavityflow_cuda_amd", "csrc"),
                    os.path.join(ROOT, "tests", "step_options_host.cpp"), "-o", exe], check=True)
    rows = "\n".join("%d %d %d %d %d %d %d %d %d" % (PRECISIONS[r[0]], *r[1], *r[2:6], len(r) > 8)
                     for r in ROWS)
    out = subprocess.run([exe], input=rows, capture_output=True, text=True, timeout=60)
    assert out.returncode == 0
    got = [tuple(int(v) for v in line.split()) for line in out.stdout.splitlines()]
    assert len(got) == len(ROWS)
    wrong = [(row, options) for row, options in zip(ROWS, got) if options != row[6:8]]
    assert not wrong
