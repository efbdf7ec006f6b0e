"""Ordering of streams of several devices, over a model of the runtime (built from
the sources, no GPU)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "opentelemac_amd", "csrc")


def test_streams_of_any_device_are_ordered(tmp_path):
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", CSRC,
                    "-I", "/opt/rocm/include", os.path.join(HERE, "stream_order_check.cpp"),
                    "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.stdout == "ok\n", out.stdout
