"""What the split loop's launchers ask for at populations that no one dispatch holds
(launch_shapes.cpp, the host part of the kernels' file on a stand-in runtime).
"""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "deac-cpp_amd", "csrc")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")
HIPCC = "/opt/rocm/bin/hipcc"


def test_dispatches_hold_their_threads(tmp_path):
    flags = ["-O1", "-std=c++17", "-ffp-contract=off", f"-I{CSRC}", f"-I{INCLUDE}", "-I/opt/rocm/include"]
    objects = []
    for src, how in ((os.path.join(CSRC, "split_kernels.hip"), [HIPCC, "--offload-arch=gfx950", "--offload-host-only"]),
                     (os.path.join(HERE, "launch_shapes.cpp"), ["g++", "-D__HIP_PLATFORM_AMD__"])):
        objects.append(str(tmp_path / (os.path.basename(src) + ".o")))
        subprocess.run([*how, *flags, "-fPIC", "-c", src, "-o", objects[-1]], check=True)
    exe = str(tmp_path / "launch_shapes")
    # the device code is left out, and the symbol that would hold it
    subprocess.run(["g++", *objects, "-Wl,--unresolved-symbols=ignore-all", "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
