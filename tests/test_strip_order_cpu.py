"""The order in which the screen passes take their tiles (vpt_tiles.h): a
permutation of the tiles whose pixel counts size the GI pass's queues.  Image
sizes around a tile, fewer than 8 tile columns, 8 and its multiples, and
widths whose last strip takes the remaining columns; the denoisers' order on
both sides of 256 tiles, with a narrow last column and without."""
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
ROOT = HERE.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_strip_order(tmp_path):
    exe = tmp_path / "strip_check"
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{ROOT / 'include'}", f"-I{ROOT / 'voxelpathtracer_amd' / 'csrc'}",
                    str(HERE / "native" / "strip_check.cpp"), "-o", str(exe)], check=True)
    sizes = [(1, 1), (16, 16), (17, 15), (15, 700), (111, 33), (112, 64), (113, 65), (127, 1), (128, 128), (129, 97),
             (320, 180), (512, 128), (513, 128), (7, 4000), (33, 1100), (260, 241), (1924, 1080), (333, 97), (255, 256), (367, 41), (1920, 1080), (1999, 1081), (16384, 3), (3, 16384)]
    r = subprocess.run([str(exe), *[str(v) for s in sizes for v in s]], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "0 mismatches", r.stdout
