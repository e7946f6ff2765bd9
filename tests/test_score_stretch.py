"""How the persistent scorer cuts the units of all rows into stretches, compiled for the host: every unit once, as evenly over
the XCDs as over the workgroups, and no stretch over a row's end where rows and stretches divide."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "socket_amd", "csrc")


@pytest.fixture(scope="module")
def stretch(tmp_path_factory):
    d = tmp_path_factory.mktemp("stretch")
    (d / "s.cpp").write_text('#include "score_stretch.h"\nextern "C" uint64_t at(uint32_t t, uint32_t g, uint32_t n) {\n'
                             "  const ScoreStretch s = score_stretch(t, g, n);\n  return (uint64_t)s.start << 32 | s.size;\n}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I" + CSRC, str(d / "s.cpp"), "-o", str(d / "s.so")], check=True)
    at = ctypes.CDLL(str(d / "s.so")).at
    at.restype = ctypes.c_uint64
    at.argtypes = [ctypes.c_uint32] * 3
    return lambda t, g, n: divmod(at(t, g, n), 1 << 32)


@pytest.mark.parametrize("groups", [1, 2, 8, 250, 256, 304, 65535])
def test_every_unit_once_and_evenly(stretch, groups):
    for total in [0, 1, 7, 8, 128, 376, 1250, 4097, 65536, 999983, 2 ** 31 - 1, 2 ** 32 - 1]:
        some = range(groups) if groups < 1000 else [0, 1, 2, 999, 32767, 32768, 65533, 65534]
        for g in some:
            start, size = stretch(total, g, groups)
            assert start == total * g // groups and start + size == total * (g + 1) // groups, (total, g)


def test_few_units_use_all_xcds(stretch):
    for total in range(1, 2048):
        # 256 workgroups, numbered XCD by XCD
        per_xcd = [sum(stretch(total, x * 32 + i, 256)[1] for i in range(32)) for x in range(8)]
        assert sum(per_xcd) == total and max(per_xcd) - min(per_xcd) <= 1, (total, per_xcd)


def test_stretches_end_with_rows(stretch):
    # 8 rows of 47 units over 256 workgroups: 32 to a row
    for g in range(256):
        start, size = stretch(376, g, 256)
        assert size == 0 or start // 47 == (start + size - 1) // 47
