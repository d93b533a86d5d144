"""The launch shapes that the autotuner times (launch_shape.h, compiled for
the CPU): the one a handle starts with is among them, once, and all fit the
LDS of a workgroup."""

from __future__ import annotations

import ctypes
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
LDS = 160 * 1024


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("shape") / "liblaunch_shape.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", str(ROOT / "tests/host/launch_shape.cpp"), "-o", str(so)],
                   check=True)
    return ctypes.CDLL(str(so))


def _candidates(lib, nq, block, levels):
    buf = (ctypes.c_int * 64)()
    n = lib.ls_candidates(LDS, nq, block, levels, buf, 32)
    assert 0 < n <= 32
    return [(buf[2 * i], buf[2 * i + 1]) for i in range(n)]


# a workgroup of 256 with half a CU's LDS (no, one, two passives), one
# wavefront with a share of it, shapes that are in the range anyway
@pytest.mark.parametrize("nq,block,levels", [(3, 256, 13), (4, 256, 10), (5, 256, 8), (5, 64, 21), (8, 64, 5), (3, 64, 0)])
def test_the_starting_shape_competes(lib, nq, block, levels):
    c = _candidates(lib, nq, block, levels)
    assert c[0] == (block, levels) and len(set(c)) == len(c)
    assert all(b * m * nq * 8 <= LDS for b, m in c)
    rest = {(b, m) for b in (64, 128, 256) for m in (0, 4, 8, 12, 16, 24, 32) if b * m * nq * 8 <= LDS}
    assert rest <= set(c)
