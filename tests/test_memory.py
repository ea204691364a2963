"""Device allocations give back spare buffers before they fail (csrc/memory.hip),
over a stand-in for the HIP calls (memory_check.cpp): a first allocation that
runs out of memory, buffers in use by this and by other threads, two devices."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "lbm_mirror_amd", "csrc")


def test_spare_buffers_go_before_an_allocation_fails(tmp_path):
    exe = str(tmp_path / "memory_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I", CSRC, os.path.join(HERE, "memory_check.cpp"), "-x", "c++",
                    os.path.join(CSRC, "memory.hip"), "-o", exe, "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
