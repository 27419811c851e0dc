"""CPU: the pinned ring whole snapshots go through (csrc/bg_snapshot.h), compiled for the host over a
stand-in for the HIP calls it makes."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_snapshot_ring(tmp_path):
    exe = str(tmp_path / "snapshot_ring")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(HERE, "..", "bitgpu_amd", "csrc"), os.path.join(HERE, "snapshot_ring.cpp"),
                    "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.stdout == "ok\n", r.stdout + r.stderr
