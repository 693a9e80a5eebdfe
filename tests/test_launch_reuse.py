"""Which calls of a batch run eagerly, are captured into a graph or replay it
(nkr-zkp_amd/csrc/launch_reuse.h), compiled for the CPU: above all, the call
after one that failed is eager, since the failed one may have left the work
buffers without the layout a capture relies on."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def reuse_bin(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("needs g++")
    out = str(tmp_path_factory.mktemp("reuse") / "launch_reuse_check")
    subprocess.run([cxx, "-O1", "-std=c++17", "-Wall", "-Werror", "-I" + os.path.join(ROOT, "nkr-zkp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "launch_reuse_check.cpp"), "-o", out], check=True)
    return out


OK, FAIL, OFF = "call 1 ok ", "call 1 fail ", "call 0 ok "
WALKS = {
    "repeat": ([OK + "1 2"] * 4, "eager capture replay replay"),
    "other key": ([OK + "1 2", OK + "1 2", OK + "2 1", OK + "1 2", OK + "1 2", OK + "1 2"],
                  "eager capture eager eager capture replay"),
    "shorter key": ([OK + "1 2", OK + "1", OK + "1", OK + "1"], "eager eager capture replay"),
    # a failed eager call: the next one may not be captured
    "eager fails": ([FAIL + "1", OK + "1", OK + "1", OK + "1"], "eager eager capture replay"),
    "eager fails twice": ([OK + "9", FAIL + "1", FAIL + "1", OK + "1", OK + "1"], "eager eager eager eager capture"),
    # a failed capture: no graph, and eager again
    "capture fails": ([OK + "1", FAIL + "1", OK + "1", OK + "1", OK + "1"], "eager capture eager capture replay"),
    # a failed replay leaves the graph, which refers to buffers of its own layout
    "replay fails": ([OK + "1", OK + "1", FAIL + "1", OK + "1"], "eager capture replay replay"),
    "not allowed": ([OFF + "1", OFF + "1", OK + "1", OK + "1"], "eager eager capture replay"),
    "dropped": ([OK + "1", OK + "1", "drop", OK + "1", OK + "1"], "eager capture drop capture replay"),
    "buffers gone": ([OK + "1", OK + "1", "forget", OK + "1", OK + "1"], "eager capture forget eager capture"),
    "first call without a key": ([OK, OK], "eager capture"),
}


@pytest.mark.parametrize("name", WALKS)
def test_modes(reuse_bin, name):
    steps, want = WALKS[name]
    res = subprocess.run([reuse_bin], input="\n".join(steps) + "\n", capture_output=True, text=True, check=True)
    assert res.stdout.split() == want.split()
