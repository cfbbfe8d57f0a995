"""Host check of the tasks of the ray walks (WalkPlan in
bonxai_amd/csrc/bxg_walk.h): every segment of every batch of rays once, and
spread over the XCDs."""
import os
import shutil
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_every_segment_is_walked_once():
    with tempfile.TemporaryDirectory() as tmp:
        exe = os.path.join(tmp, "walk_plan_check")
        subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "bonxai_amd", "csrc"),
                        os.path.join(HERE, "walk", "walk_plan_check.cpp"), "-o", exe], check=True)
        out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
        assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout + out.stderr
