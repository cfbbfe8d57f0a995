"""Host check of the leaf pass's walk (LeafWalk in
bonxai_amd/csrc/bxg_walk.h): the leaves of whole rays and of parts of them, for
every leaf and inner grid size, on both sides of the 32-bit limit, against the
leaves of the ray's cells one by one."""
import os
import shutil
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_leaves_match_cells():
    with tempfile.TemporaryDirectory() as tmp:
        exe = os.path.join(tmp, "leaf_walk_check")
        subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "bonxai_amd", "csrc"),
                        os.path.join(HERE, "walk", "leaf_walk_check.cpp"), "-o", exe], check=True)
        out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
        assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout + out.stderr
