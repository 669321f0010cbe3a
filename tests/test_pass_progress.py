"""The records by which a pass's iterations report to the host (naivetrace_amd/csrc/pass_progress.hpp), on
the CPU: an iteration waits for its own report only, also when a pass before it was left unfinished."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_reports_belong_to_their_pass(tmp_path):
    exe = str(tmp_path / "pass_progress_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", os.path.join(ROOT, "tests", "cpp", "pass_progress_check.cpp"), "-o", exe],
                   check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
