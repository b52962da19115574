"""The rule by which an FP64 batch takes its launch form, on the CPU
(tests/host_check/batch_form_check.cpp)."""
import os
import subprocess

TESTS = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(TESTS), "dgcuda_amd", "csrc")
HERE = os.path.join(TESTS, "host_check")


def test_batch_form(tmp_path):
    exe = str(tmp_path / "batch_form_check")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", HERE, "-I", CSRC, os.path.join(HERE, "batch_form_check.cpp"),
                    "-o", exe], check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0 and "batch form ok" in r.stdout, r.stdout
