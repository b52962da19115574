"""Admission counts at least what a resident solve allocates, on the CPU
(tests/host_check/solve_bytes_check.cpp)."""
import os
import subprocess

TESTS = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(TESTS), "dgcuda_amd", "csrc")
HERE = os.path.join(TESTS, "host_check")


def test_counted_bytes_cover_the_allocations(tmp_path):
    exe = str(tmp_path / "solve_bytes_check")
    subprocess.run(["g++", "-std=c++17", "-DDG_GLOBAL=", "-I", HERE, "-I", CSRC,
                    os.path.join(HERE, "solve_bytes_check.cpp"), "-o", exe],
                   check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0 and "solve bytes ok" in r.stdout, r.stdout
