"""The host threads of one call (gsplat_tt_amd/csrc/host_threads.h) on the CPU:
tests/host_threads_check.cpp is built with g++ against the header and run, plain and,
where g++ has its runtime, under ThreadSanitizer."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
INC = os.path.join(os.path.dirname(HERE), "gsplat_tt_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("extra", [[], ["-fsanitize=thread"]], ids=["plain", "tsan"])
def test_host_threads(tmp_path, extra):
    if extra:
        probe = subprocess.run(["g++", *extra, "-x", "c++", "-", "-o", str(tmp_path / "probe")],
                               input="int main(){return 0;}", text=True, capture_output=True)
        if probe.returncode != 0 or subprocess.run([str(tmp_path / "probe")]).returncode != 0:
            pytest.skip("g++ has no ThreadSanitizer runtime here")
    exe = str(tmp_path / "host_threads_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-Wextra", "-Werror", "-I", INC,
                    os.path.join(HERE, "host_threads_check.cpp"), "-o", exe, "-pthread", *extra],
                   check=True, timeout=120)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stderr[-2000:]
