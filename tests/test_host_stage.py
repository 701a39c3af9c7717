"""Copies of results to the caller's memory (HostStage) with a stand-in for the runtime,
whose calls are counted and can be made to fail: which copies go through the pinned
pieces and which directly. tests/host_stage.cpp does the checks, one name each."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("stage") / "host_stage")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wextra", "-pthread", f"-I{ROOT}/pdekit_amd/csrc/hip", "-o", exe,
                    f"{ROOT}/tests/host_stage.cpp"], check=True)
    return exe


@pytest.mark.parametrize("name", ["sizes", "pinned", "made_late", "failures"])
def test_host_stage(program, name):
    out = subprocess.run([program, name], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
