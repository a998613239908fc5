"""Which steps of a plan share a launch (no GPU).

A launch may run the steps after its own only where each starts at the level
the one before it ended with; a custom dispatcher may record others.
tests/host/plan_launches.cpp runs the library's executor on such plans with
launchers of its own, which only note what they are asked for.
"""
import os
import shutil
import subprocess

import pytest

from vk_compute_mipmaps_amd import build

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")


@pytest.mark.skipif(not (os.path.exists(build.hipcc()) or shutil.which("hipcc")), reason="needs hipcc")
def test_steps_share_a_launch_only_in_order():
    out = os.path.join(HERE, "_build", "plan_launches")
    os.makedirs(os.path.dirname(out), exist_ok=True)
    if not os.path.exists(build.LIB_PATH):
        build.build_library()
    # The program's own launchers are found before the library's.
    cmd = [build.hipcc(), "--offload-arch=gfx950", "-O1", "-std=c++17", "-x", "hip", "-I", build.INCLUDE, "-I", build.CSRC,
           os.path.join(HERE, "plan_launches.cpp"), "-o", out, "-L", build.LIB_DIR, "-lnvpro_pyramid_hip",
           f"-Wl,-rpath,{build.LIB_DIR}"]
    made = subprocess.run(cmd, capture_output=True, text=True)
    assert made.returncode == 0, made.stderr[-4000:]
    run = subprocess.run([out], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout + run.stderr
