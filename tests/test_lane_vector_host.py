"""The Euler lane body in the vector layout (p <= 3) against the general lane
body on the CPU: same state, mesh and RK operands through both, every stage
kind, with and without boundary sides, element counts that divide by no
workgroup, under AddressSanitizer with buffers of exactly the device sizes
(tests/host_check/lane_vec_check.cpp)."""
import os
import subprocess

import pytest

import dgcuda_amd as dg

TESTS = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(TESTS), "dgcuda_amd", "csrc")
HERE = os.path.join(TESTS, "host_check")
GOLD = os.path.join(TESTS, "golden")
CLANG = "/opt/rocm/llvm/bin/clang++"


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    if not os.path.exists(CLANG):
        pytest.skip("clang++ with AddressSanitizer not available")
    exe = str(tmp_path_factory.mktemp("host_check") / "lane_vec_check")
    cmd = [CLANG, "-std=c++17", "-O0", "-fsanitize=address", "-DDG_GLOBAL=", "-I", HERE, "-I", CSRC,
           os.path.join(HERE, "lane_vec_check.cpp")] + \
          [os.path.join(CSRC, f) for f in ("dg_geometry.cpp", "dg_mesh.cpp", "dg_tables.cpp")] + ["-o", exe]
    subprocess.run(cmd, check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    return exe


@pytest.mark.parametrize("mesh", ["periodic", "boundary"])
@pytest.mark.parametrize("p", [1, 2, 3])
@pytest.mark.parametrize("prec", [0, 1])
def test_vector_body_equals_general_body(harness, tmp_path, mesh, p, prec):
    path = os.path.join(GOLD, "sv1refined.pmsh")
    if mesh == "periodic":
        path = str(tmp_path / "periodic.pmsh")
        dg.Mesh.periodic_jittered(11, 9, 0.0, 10.0, 0.0, 8.0, 0.1, 3).write_pmsh(path)
    r = subprocess.run([harness, path, str(p), str(prec)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                       text=True, timeout=120)
    assert r.returncode == 0 and "bodies agree" in r.stdout, r.stdout[-3000:]
