"""The mark of the vectors that workgroups of one launch hand to one another, on the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_share_mark(tmp_path):
    exe = str(tmp_path / "share_mark_check")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
                        "-fno-sanitize-recover=all", "-I", os.path.join(ROOT, "onsas.jl_amd", "csrc"),
                        os.path.join(ROOT, "tests", "host", "share_mark_check.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok 1\n", r.stdout + r.stderr
