"""The rules that choose how a frame's tile lists are made (gsplat_tt_amd/csrc/tile_plan.h)
on the CPU: tests/tile_plan_check.cpp is built with g++ against the header and run."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
INC = os.path.join(os.path.dirname(HERE), "gsplat_tt_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_tile_plan(tmp_path):
    exe = str(tmp_path / "tile_plan_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-I", INC,
                    os.path.join(HERE, "tile_plan_check.cpp"), "-o", exe], check=True,
                   timeout=120)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stderr
