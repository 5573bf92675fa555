"""The host code of the engine and the batch on a stand-in for the HIP runtime
(host_runtime.cpp): what it asks for, and what it leaves behind when an
allocation or a launch fails.  No device, no kernel.
"""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "deac-cpp_amd", "csrc")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_runtime") / "host_runtime")
    sources = [os.path.join(HERE, "host_runtime.cpp")] + [
        os.path.join(CSRC, f) for f in ("engine.cpp", "batch.cpp", "precision.cpp", "host_model.cpp")]
    subprocess.run(["g++", "-O1", "-std=c++20", "-ffp-contract=off", "-march=x86-64-v3", "-D__HIP_PLATFORM_AMD__",
                    f"-I{CSRC}", f"-I{INCLUDE}", "-I/opt/rocm/include", *sources, "-lpthread", "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["status_memory", "long_histories", "host_memory_runs_out", "launches_fail",
                                      "device_memory_runs_out"])
def test_host_runtime(program, scenario):
    r = subprocess.run([program, scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
