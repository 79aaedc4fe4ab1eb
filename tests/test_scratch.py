"""Which scratch buffer a product takes (csrc/scratch.h), on the CPU: buffers
of streams, of threads and of captured graphs never meet."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_scratch_rules(tmp_path):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no host compiler")
    exe = str(tmp_path / "scratch_test")
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread",
                    "-I", os.path.join(ROOT, "tinyoai_amd", "csrc"),
                    os.path.join(ROOT, "tests", "scratch_test.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
