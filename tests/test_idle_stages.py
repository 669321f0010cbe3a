"""The pool of idle ray-query stages (naivetrace_amd/csrc/idle_stages.hpp) on the CPU: a small query never
takes the large queries' stage, gets the smallest that fits, and giving a stage back cannot throw (it
happens in a destructor, also when memory has run out)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_idle_stages(tmp_path):
    exe = str(tmp_path / "idle_stages_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", os.path.join(ROOT, "tests", "cpp", "idle_stages_check.cpp"), "-o", exe],
                   check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
