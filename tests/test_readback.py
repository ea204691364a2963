"""Read-back (csrc/readback.hip) over a stand-in for the HIP calls
(readback_check.cpp), also where no pinned memory is to be had."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "lbm_mirror_amd", "csrc")


def test_read_back_with_and_without_pinned_memory(tmp_path):
    exe = str(tmp_path / "readback_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", CSRC,
                    os.path.join(HERE, "readback_check.cpp"), "-x", "c++", os.path.join(CSRC, "readback.hip"),
                    "-o", exe, "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
