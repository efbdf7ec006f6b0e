"""Turns of processes on one GPU (built from the sources, no GPU)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "opentelemac_amd", "csrc")


def test_one_process_at_a_time(tmp_path):
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, os.path.join(HERE, "turn_check.cpp"),
                    "-o", exe], check=True)
    files = tmp_path / "files"
    files.mkdir()
    out = subprocess.run([exe, str(files)], capture_output=True, text=True, timeout=120)
    assert out.stdout == "ok\n", (out.stdout, out.stderr)
