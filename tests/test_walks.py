"""Bounds of the direct solve's walks (kmst_walks.hpp), on the CPU."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "kamsta_amd", "csrc")


def test_a_walk_round_a_cycle_ends(tmp_path):
    exe = str(tmp_path / "check_walks")
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", CSRC, "-o", exe,
                        os.path.join(HERE, "host", "check_walks.cpp")],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "ok (walks)" in r.stdout, r.stdout + r.stderr
