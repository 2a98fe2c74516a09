"""The replay of a captured graph as its kernel launches (csrc/g4_graph_replay.h), on the CPU: a C++
driver with fake launch, event and drain calls checks that a launch that fails behind others leaves
the event recorded that g4_graph_destroy waits for, and that a replay whose event cannot be recorded
waits for the stream."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "gemma4-webgpu-engine_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_partial_replays_are_marked(tmp_path):
    exe = tmp_path / "replay_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC,
                    os.path.join(HERE, "graph_replay_check.cc"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
