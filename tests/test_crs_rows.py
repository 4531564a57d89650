"""The look over a CRS row pointer before an upload (csrc/crs_rows.h), built
for the host: it names the first row at which the pointer decreases, whatever
the size of the step (steps of more than 2^31 wrap in 32 bits), and the
longest row."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from tests.conftest import REPO

BIG = 2_000_000_000


@pytest.fixture(scope="module")
def crs_rows(tmp_path_factory):
    d = tmp_path_factory.mktemp("crs_rows")
    src, lib = str(d / "shim.cpp"), str(d / "shim.so")
    with open(src, "w") as f:
        f.write('#include "crs_rows.h"\n'
                'extern "C" int rows(int n, const int *ptr, int *longest) {\n'
                "  return cghip::crs_rows(n, ptr, longest);\n}\n")
    subprocess.run(["g++", "-std=c++17", "-O3", "-shared", "-fPIC",
                    "-I" + os.path.join(REPO, "cgxx_amd", "csrc"), "-o", lib, src], check=True)
    L = ctypes.CDLL(lib)

    def call(ptr):
        ptr = np.ascontiguousarray(ptr, np.int32)
        longest = ctypes.c_int(-7)
        return L.rows(ptr.size - 1, ptr.ctypes.data_as(ctypes.c_void_p), ctypes.byref(longest)), longest.value

    return call


@pytest.mark.parametrize("ptr, row", [
    ([0, BIG, -BIG, 0, 4], 1),
    ([0, BIG, -BIG, 100], 1),
    ([0, 1, BIG, -BIG, 4], 2),
    ([0, 4, 3, 4], 1),
    ([0, -1, 4], 0),
    ([0, 5, 4], 1),
    ([0, 2**31 - 1, -2**31, 0], 1),
    ([0] * 300 + [BIG, -BIG, 0] + [7] * 300, 300),
])
def test_decrease_is_found(crs_rows, ptr, row):
    assert crs_rows(ptr)[0] == row


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1000])
def test_longest_row(crs_rows, n):
    length = np.random.default_rng(n).integers(0, 2_000_000, n)
    ptr = np.concatenate([[0], np.cumsum(length)])
    assert ptr[-1] < 2**31
    assert crs_rows(ptr) == (-1, length.max())
    assert crs_rows(np.zeros(n + 1)) == (-1, 0)
    assert crs_rows(np.concatenate([np.zeros(n), [2**31 - 1]])) == (-1, 2**31 - 1)


@pytest.mark.parametrize("seed", range(20))
def test_any_pointer(crs_rows, seed):
    ptr = np.random.default_rng(seed).integers(-2**31, 2**31, 40)
    down = np.flatnonzero(np.diff(ptr) < 0)
    assert crs_rows(ptr)[0] == down[0]
