"""Copying of the pinned read-back (nanogi_amd/csrc/ngi_copy.h), compiled and
run on the host by tests/copy_check.cpp.
"""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_chunks_are_copied_once_and_nobody_waits_for_a_late_helper(tmp_path):
    exe = tmp_path / "copy_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-I", os.path.join(ROOT, "nanogi_amd", "csrc"),
                    os.path.join(ROOT, "tests", "copy_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
