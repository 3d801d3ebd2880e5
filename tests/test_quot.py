"""Quotients of the ray set-up (nanogi_amd/csrc/ngi_quot.h): wherever the
traversal takes them, the multiply-adds give the bits of the IEEE division.
tests/quot_check.cpp compiles the same header on the host.
"""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_multiply_adds_are_the_division(tmp_path):
    exe = tmp_path / "quot_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-I", os.path.join(ROOT, "nanogi_amd", "csrc"),
                    os.path.join(ROOT, "tests", "quot_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith("ok ") and int(r.stdout.split()[1]) > 100000000
