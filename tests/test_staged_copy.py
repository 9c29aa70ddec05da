"""The threads of large copies to the host (csrc/staged_copy.h), over plain memory: sizes around the
chunk and the number of workers, and every call of the link failing once.  CPU only."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_staged_copy_is_whole_and_reports_errors(tmp_path):
    run = lambda cmd: subprocess.run(cmd, cwd=tmp_path, capture_output=True, text=True, timeout=120)
    r = run(["g++", "-O1", "-std=c++17", "-pthread", "-I", os.path.join(ROOT, "specfwat_amd", "csrc"), "-o", "check",
             os.path.join(ROOT, "tests", "staged_copy_check.cpp")])
    assert r.returncode == 0, r.stderr
    r = run([str(tmp_path / "check")])
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
