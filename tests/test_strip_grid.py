"""The strip kernel's block order (csrc/g4_strip_grid.h), on the CPU: every strip is one block's, and no XCD
gets more strips than it has CUs (one more would be a second round for the whole call)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "gemma4-webgpu-engine_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_strips_cover_the_output_in_one_round(tmp_path):
    exe = tmp_path / "strip_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC,
                    os.path.join(HERE, "strip_grid_check.cc"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
