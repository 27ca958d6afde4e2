"""The state downloads through pinned buffers (genesis6_amd/csrc/g6_stage.h)
on the host, with a stand-in for the HIP runtime that knows which device an
event and a stream belong to and counts the bytes it copies
(tests/stage_host)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("stage") / "stage")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I" + os.path.join(HERE, "stage_host"),
                    "-I" + os.path.join(HERE, "..", "genesis6_amd", "csrc"),
                    os.path.join(HERE, "stage_host", "main.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("name", ["devices", "ranges", "busy"])
def test_staged_download(program, name):
    r = subprocess.run([program, name], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
