"""The launch options that whole-domain steps choose, compiled for the host: every
line of the choice at sizes on both of its sides, and that the sizes of the GPU tests
of the choice lie in the part that each is there for."""
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
    # all within the Infinity Cache
    ("f32", (86, 83, 81), 0, WALL, 0, 0, 0, X | W2), ("f64", (70, 69, 67), 0, WALL, 0, 0, 0, X | W3),
    ("f16s", (107, 103, 101), 0, WALL, 0, 0, P, P | X | W4),
    ("f16c", (107, 103, 101), 0, WALL, 0, 0, P, P | X | W4),
    ("bf16s", (107, 103, 101), 0, WALL, 0, 0, P, P | X | W4),
    # only the state itself
    ("f32", (86, 83, 81), 0, WALL, 0, 348, W3, BIG | W4),
    ("f64", (70, 69, 67), 0, WALL, 0, 348, W2, W3),
    ("f16s", (107, 103, 101), 0, WALL, 0, 348, P | W4, P | X | W3),
    ("f16c", (107, 103, 101), 0, WALL, 0, 348, P | W4, P | W4),
    # fits, but not with the others: round and round, to and fro
    ("f32", (86, 83, 81), 0, WALL, 348, 348, NT | W2, W2),
    ("f32", (86, 83, 81), 0, WALL, 220, 348, W2, X | W3 | REV),
    ("f64", (70, 69, 67), 0, WALL, 220, 500, W2, X | W3 | REV),
    ("f16s", (107, 103, 101), 0, WALL, 348, 348, P | NT | W3, P | X | W4),
    ("f16s", (107, 103, 101), 0, GHOST, 348, 348, P | W3, P | X | W4),
    # nontemporal stores left nothing in the cache, whatever came between
    ("f32", (86, 83, 81), 0, WALL, 0, 348, NT | W2, W2, 1),
    ("f64", (70, 69, 67), 0, WALL, 0, 0, NT | W2, W2, 1),
    ("f16s", (107, 103, 101), 0, WALL, 0, 0, P | NT | W3, P | X | W4, 1),
    ("f16s", (190, 187, 193), 0, WALL, 0, 0, P | NT | W4, P | W4, 1),
    # larger than the cache
    ("f32", (151, 149, 150), 0, WALL, 0, 0, W4, BIG | W4 | REV),
    ("f32", (229, 186, 141), 1, WALL, 0, 0, W4, BIG | W4 | REV),
    ("f32", (229, 186, 141), 1, WALL, 0, 348, W2, BIG | W4 | REV),
    ("f32", (217, 217, 217), 0, WALL, 0, 0, W2, BIG | W4 | REV),
    ("f32", (275, 275, 275), 0, WALL, 0, 0, W2, BIG | W4 | REV),
    ("f32", (281, 280, 279), 0, WALL, 0, 0, W2, LDS | W4 | REV),
    ("f32", (350, 345, 345), 0, WALL, 0, 0, NT | W2, LDS | W4 | REV),
    ("f64", (150, 147, 139), 0, WALL, 0, 0, W2, W2 | REV),
    ("f64", (227, 226, 225), 0, WALL, 0, 0, W2, W2 | REV),
    ("f64", (233, 232, 231), 0, WALL, 0, 0, W2, LDS | W2 | REV),
    ("f64", (280, 271, 275), 0, WALL, 0, 0, NT | W2, LDS | W2 | REV),
    ("f16s", (190, 187, 193), 0, WALL, 0, 0, P | NT | W4, P | W4),
    ("f16c", (221, 219, 220), 0, WALL, 0, 0, P | NT | W4, P | W4),
    ("f16s", (190, 187, 193), 0, WALL, 0, 348, P | W3, P | W4 | REV),
    ("f16s", (205, 203, 199), 1, WALL, 0, 0, P | W3, P | W4 | REV),
    ("bf16s", (241, 260, 277), 1, WALL, 0, 0, P | W3, P | W4 | REV),
    ("bf16s", (300, 290, 277), 1, WALL, 0, 0, P | NT | W3, P | W3 | REV),
    ("f16s", (321, 319, 320), 0, WALL, 0, 0, P | NT | W3, P | W3 | REV),
    ("f16c", (321, 319, 320), 0, WALL, 0, 0, P | NT | W4, P | W4 | REV),
    # exchanged faces: never nontemporal
    ("f16s", (190, 187, 193), 0, GHOST, 0, 0, P | W3, P | W4 | REV),
    ("f16c", (321, 319, 320), 0, GHOST, 0, 0, P | W3, P | W4 | REV),
    ("f32", (281, 280, 279), 0, GHOST, 0, 0, W2, LDS | W4 | REV),
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
