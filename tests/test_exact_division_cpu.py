"""The denoisers' short forms of divisions, exp and log (vpt_short_math.h, the
code that the kernels compile) against the full ones, built for the CPU: fmaf
there is exact, as the GPU's v_fma_f32 is.  x / 3 of the shadow filter is
compared with the IEEE division for every float in [0, 2]."""
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


def _check(tmp_path, name):
    exe = tmp_path / name
    # -ffp-contract=off: products and sums round as written
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-mfma", "-pthread",
                    f"-I{HERE.parent / 'include'}", f"-I{HERE.parent / 'voxelpathtracer_amd' / 'csrc'}",
                    str(HERE / "native" / f"{name}.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
    assert r.stdout.strip().endswith("0 mismatches")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_div3_unit_equals_division_on_0_2(tmp_path):
    _check(tmp_path, "div3_check")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_denoiser_exp_and_log_equal_the_full_ones(tmp_path):
    _check(tmp_path, "exp_log_check")
