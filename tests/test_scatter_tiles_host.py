"""The tile maps of the MFMA scatter under AddressSanitizer.

csrc/projector_maps.h is compiled with g++ -fsanitize=address,undefined into a small
driver (tests/asan/scatter_tiles_check.cpp): every voxel of every atom is in exactly
one row of its atom at its point's place, all other places are empty, every tile has
a row.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "qumasun-workshop-template_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_scatter_tiles_under_asan(tmp_path):
    exe = str(tmp_path / "scatter_tiles_check")
    cmd = ["g++", "-std=c++17", "-O1", "-g", "-fno-omit-frame-pointer",
           "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
           f"-I{CSRC}", os.path.join(HERE, "asan", "scatter_tiles_check.cpp"), "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, f"build failed:\n{' '.join(cmd)}\n{r.stdout}{r.stderr}"
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, f"{r.stdout}{r.stderr}"
    assert "cases ok" in r.stdout
