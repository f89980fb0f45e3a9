"""The rules of the null stream's kept memory, compiled for the host: reuse,
the limit and the order in which blocks go, give-back on failure, the drop,
blocks of several devices, many free blocks of one size, how much larger
than asked for a block may be, and calls without host memory."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("kept") / "kept_memory_test")
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "engine_amd", "csrc"),
           os.path.join(ROOT, "tests", "cpp", "kept_memory_test.cpp"), "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return out


@pytest.mark.parametrize("check", ["reuse", "limit", "failure", "drop", "devices", "many", "excess", "host_memory"])
def test_kept_memory(exe, check):
    r = subprocess.run([exe, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert f"{check} ok" in r.stdout
