"""Scratch memory of the general lane kernels, as the compiler recorded it in
the built library: sums left to be formed behind a branch spilled up to 9 KB
a lane.  The bounds are what the kernels take when each face's sums are formed
in place (Euler at p = 4, 5 in FP64 does not fit the registers in any order).
CPU only."""
import re
import struct
import subprocess

import pytest

import dgcuda_amd as dg

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


@pytest.fixture(scope="module")
def scratch(tmp_path_factory):
    """Mangled kernel name -> bytes of scratch per lane."""
    d = open(dg.LIB_PATH, "rb").read()
    out, at = {}, d.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        (n,), pos = struct.unpack_from("<Q", d, at + 24), at + 32
        for _ in range(n if n < 8 else 0):  # (the name alone may stand elsewhere)
            off, size, length = struct.unpack_from("<QQQ", d, pos)
            if b"gfx950" in d[pos + 24:pos + 24 + length]:
                f = tmp_path_factory.mktemp("co") / "code.o"
                f.write_bytes(d[at + off:at + off + size])
                notes = subprocess.run([READELF, "--notes", str(f)], check=True, stdout=subprocess.PIPE,
                                       text=True).stdout
                names = re.findall(r"\.name: +(_Z\S+)", notes)
                sizes = re.findall(r"\.private_segment_fixed_size: +(\d+)", notes)
                assert len(names) == len(sizes)
                out.update(zip(names, map(int, sizes)))
            pos += 24 + length
        at = d.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)
    return out


# (variables, order, precision) -> bytes
LANE_BOUNDS = {(1, 5, "d"): 128, (1, 5, "f"): 64, (4, 4, "f"): 64, (4, 5, "f"): 128, (4, 4, "d"): 3100, (4, 5, "d"): 4976}


def test_general_lane_kernels(scratch):
    seen = 0
    for name, size in scratch.items():
        m = re.search(r"12k_stage_valuILi(\d)ELi(\d)E([fd])", name)
        if not m:
            continue
        seen += 1
        key = (int(m[1]), int(m[2]), m[3])
        assert size <= LANE_BOUNDS.get(key, 0), (name, size)
    assert seen >= 40


def test_batch_stage_kernels(scratch):
    """Every launch form's kernel: at most a few values, kept over a run of
    items; the bodies' own values stay in registers."""
    sizes = {n: s for n, s in scratch.items() if "13k_batch_stageI" in n}
    assert len(sizes) == 40  # precisions x stages x masks
    assert max(sizes.values()) <= 128, {n: s for n, s in sizes.items() if s > 128}
