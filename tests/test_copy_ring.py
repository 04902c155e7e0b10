"""The ring of the large downloads on a device made of a thread, on the host."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("sanitizer", ["address,undefined", "thread"])
def test_copy_ring(tmp_path, sanitizer):
    exe = str(tmp_path / "copy_ring_check")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", f"-fsanitize={sanitizer}",
                        "-fno-sanitize-recover=all", "-pthread", "-I",
                        os.path.join(ROOT, "onsas.jl_amd", "csrc"),
                        os.path.join(ROOT, "tests", "host", "copy_ring_check.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
