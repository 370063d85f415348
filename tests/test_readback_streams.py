"""The threads of a read-back copy after the work queued on the caller's stream,
also where the handle names another stream in each thread: rbhip_readback.h
built for the host against a model of streams and events (cpu_streams)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HERE = os.path.join(ROOT, "tests", "cpu_streams")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("cpu_streams") / "readback")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", HERE, "-I",
                    os.path.join(ROOT, "openmm_rigidbody_plugin_amd", "csrc"), os.path.join(HERE, "readback_main.cpp"),
                    "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("per_thread", [0, 1])
@pytest.mark.parametrize("nbytes", [1, 2 << 20, (2 << 20) + 1, (4 << 20) + 8, 17 << 20])
def test_copies_follow_the_callers_work(program, nbytes, per_thread):
    out = subprocess.run([program, str(nbytes), str(per_thread)], check=True, capture_output=True, text=True, timeout=60)
    assert int(out.stdout) == 0
