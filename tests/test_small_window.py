"""The host's side of a small download ends whatever the kernel leaves in the window, and writes the caller's memory only when
every word is there; threads stand for the kernel (no GPU needed)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "spoc_amd", "csrc")
CLANG = "/opt/rocm/llvm/bin/clang++"


@pytest.mark.skipif(not os.path.exists(CLANG), reason="no clang++ in this image")
def test_words_that_come_late_or_never(tmp_path):
    exe = str(tmp_path / "small_window")
    build = subprocess.run([CLANG, "-std=c++20", "-O1", "-g", "-fsanitize=address,undefined", "-Wall", "-I" + CSRC,
                            os.path.join(HERE, "host_sanitizers", "small_window.cpp"), "-lpthread", "-o", exe],
                           capture_output=True, text=True)
    assert build.returncode == 0, build.stderr[-3000:]
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and "small window ok" in run.stdout, run.stdout + run.stderr
