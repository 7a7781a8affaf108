"""The pinned-ring copy to host memory (gn_copy.h) on the CPU, its HIP calls
replaced by host ones (tests/native): every byte arrives for segments that are
cut and packed, and an allocation, thread, copy or wait that fails at any
point ends in an exception or a finished copy, never in a terminated process
or a hang."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_host_copy_survives_failures(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "host_copy_check"
    subprocess.run([cxx, "-std=c++17", "-O1", "-g", "-I", os.path.join(HERE, "native"),
                    os.path.join(HERE, "native", "host_copy_check.cpp"), "-o", str(exe),
                    "-pthread", "-ldl", "-rdynamic"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
