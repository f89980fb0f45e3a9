"""merge_sorted's tile arithmetic, compiled for the host: lists in any order
leave every access inside them, ascending lists are cut at the merge path."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tiles_stay_inside_the_lists(tmp_path):
    exe = str(tmp_path / "merge_path_test")
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-D__host__=", "-D__device__=", "-D__forceinline__=inline",
           "-I", os.path.join(ROOT, "engine_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "merge_path_test.cpp"),
           "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "merge path ok" in r.stdout
