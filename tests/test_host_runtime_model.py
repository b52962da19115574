"""Host code between the caller and the runtime, compiled against a model of
the runtime's host side (tests/host_check/runtime) and run under sanitizers:
the replay of captured steps (dg_step_graph.h) and the copies through pinned
blocks (dg_hostcopy.cpp).  CPU only."""
import os
import subprocess

import pytest

TESTS = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(TESTS), "dgcuda_amd", "csrc")
HERE = os.path.join(TESTS, "host_check")


def run(tmp_path, name, sources, flags, *args):
    exe = str(tmp_path / name)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-DDG_GLOBAL=", "-I",
                    os.path.join(HERE, "runtime"), "-I", HERE, "-I", CSRC, os.path.join(HERE, name + ".cpp")] +
                   [os.path.join(CSRC, s) for s in sources] + flags + ["-ldl", "-o", exe],
                   check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    r = subprocess.run([exe] + list(args), stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-4000:]
    return r.stdout


@pytest.mark.parametrize("sanitizer", ["address,undefined", "thread"])
def test_step_graph(tmp_path, sanitizer):
    assert "step graphs ok" in run(tmp_path, "step_graph_check", [], ["-fsanitize=" + sanitizer])


@pytest.mark.parametrize("flags,args", [(["-fsanitize=address,undefined"], ()), (["-fsanitize=thread"], ("brief",)),
                                        (["-DNO_THREADS"], ())])
def test_host_copies(tmp_path, flags, args):
    assert "host copies ok" in run(tmp_path, "hostcopy_check", ["dg_hostcopy.cpp"], flags, *args)
