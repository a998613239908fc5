"""The tile rows of large fast steps (no GPU).

The kernels find a tile's row by multiplication.  tests/host/fast_tile_rows.cpp
runs the kernels' own expression, with the inverse the launcher makes, on the
CPU over every level width and height there can be.
"""
import os
import shutil
import subprocess

import pytest

from vk_compute_mipmaps_amd import build

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")


@pytest.mark.skipif(not (os.path.exists(build.hipcc()) or shutil.which("hipcc")), reason="needs hipcc")
def test_rows_by_multiplication_equal_the_division():
    out = os.path.join(HERE, "_build", "fast_tile_rows")
    os.makedirs(os.path.dirname(out), exist_ok=True)
    cmd = [build.hipcc(), *build.HIPCC_FLAGS, "-x", "hip", "-I", build.INCLUDE, "-I", build.CSRC,
           os.path.join(HERE, "fast_tile_rows.cpp"), "-o", out]
    made = subprocess.run(cmd, capture_output=True, text=True)
    assert made.returncode == 0, made.stderr[-4000:]
    run = subprocess.run([out], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0, run.stdout + run.stderr
