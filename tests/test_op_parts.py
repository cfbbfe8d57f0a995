"""Host check of the parts that a bucket of a bulk cell call is done in (OpPart
in bonxai_amd/csrc/bxg_op_parts.h): every cell in exactly one of them, and few
passes over buckets of many leaves or cells."""
import os
import shutil
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_parts_cover_a_bucket_once_in_few_passes():
    with tempfile.TemporaryDirectory() as tmp:
        exe = os.path.join(tmp, "op_parts_check")
        subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "bonxai_amd", "csrc"),
                        os.path.join(HERE, "walk", "op_parts_check.cpp"), "-o", exe], check=True)
        out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
        assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout + out.stderr
