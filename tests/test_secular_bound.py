"""The secular roots of the tridiagonal divide and conquer end within their bound.

csrc/secular.h runs on the GPU with a wave per root; here it is compiled with g++
-fsanitize=address,undefined into a small driver (tests/asan/secular_check.cpp) that
solves random problems one lane at a time, with the rational steps and without
them.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "qumasun-workshop-template_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_secular_roots_within_bound(tmp_path):
    exe = str(tmp_path / "secular_check")
    cmd = ["g++", "-std=c++17", "-O1", "-g", "-fno-omit-frame-pointer",
           "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
           f"-I{CSRC}", os.path.join(HERE, "asan", "secular_check.cpp"), "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, f"build failed:\n{' '.join(cmd)}\n{r.stdout}{r.stderr}"
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, f"{r.stdout}{r.stderr}"
    assert "roots ok" in r.stdout
