"""Work shared by host threads (kmst_threads.hpp, the host API's staging):
every item is done once, whichever threads the system refuses."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "kamsta_amd", "csrc")


def test_refused_threads_leave_no_work_undone(tmp_path):
    exe = str(tmp_path / "check_threads")
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-pthread", "-rdynamic", "-I", CSRC, "-o", exe,
                        os.path.join(HERE, "host", "check_threads.cpp"), "-ldl"],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "ok (threads)" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
