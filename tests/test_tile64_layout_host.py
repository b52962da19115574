"""The FP64 tile layout's placement of modes (tile64_at): every (mode,
element) of a block's variable has a place of its own inside the block, and
a lane's registers sit where its accesses read them, at every order."""
import os
import subprocess

import pytest

TESTS = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(TESTS), "dgcuda_amd", "csrc")

SRC = r"""
#include <cstdio>
#include <cstring>
#include <hip/hip_runtime.h>
#include "dg_device.h"
using namespace dgmi;
int main() {
    for (int p = 1; p <= 4; p++) {
        const int NP = n_modes(p), S = tile64_slots(NP);
        bool used[256] = {};
        for (int m = 0; m < NP; m++)
            for (int j = 0; j < 16; j++) {
                const int at = tile64_at(NP, m, j);
                if (at < 0 || at >= 16 * S || used[at]) return 1;
                used[at] = true;
                const int g = m & 3, r = m >> 2;
                // the pieces: pairs (r = 0, 1) and (2, 3) of a lane are 16 bytes, aligned
                if (NP > 8 && r < 2 && at != (g * 16 + j) * 2 + r) return 2;
                if (NP > 12 && r >= 2 && at != 128 + (g * 16 + j) * 2 + r - 2) return 3;
                if (NP > 8 && NP <= 12 && r == 2 && at != 128 + g * 16 + j) return 4;
                if (NP <= 8 && at != r * 64 + g * 16 + j) return 5;
            }
        const StateIx ix{4, NP, 64, LAYOUT_TILE64};
        if (ix.elems() != (size_t)4 * S * 64 || ix.at(3, NP - 1, 63) >= ix.elems()) return 6;
    }
    puts("placed");
    return 0;
}
"""


def test_tile64_places(tmp_path):
    clang = "/opt/rocm/llvm/bin/clang++"
    if not os.path.exists(clang):
        pytest.skip("clang++ not available")
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(SRC)
    subprocess.run([clang, "-std=c++17", "-DDG_GLOBAL=", "-I", os.path.join(TESTS, "host_check"), "-I", CSRC, str(src),
                    "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, check=True).stdout.strip() == "placed"
