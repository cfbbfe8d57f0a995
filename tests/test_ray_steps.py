"""Host check of the closed forms that start a ray mid-way (RayWalk::steps,
seek in bonxai_amd/csrc/bxg_walk.h): 32-bit arithmetic up to 32767 cells a
ray, 64-bit beyond, against the formula in 64 bits."""
import os
import shutil
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_steps_match_closed_form():
    with tempfile.TemporaryDirectory() as tmp:
        exe = os.path.join(tmp, "ray_steps_check")
        subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "bonxai_amd", "csrc"),
                        os.path.join(HERE, "walk", "ray_steps_check.cpp"), "-o", exe], check=True)
        out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
        assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout + out.stderr
