"""The width in which a small pull copies rows (csrc/row_width.h): every length, distance and place of a variable has one, and
its accesses are aligned wherever the elements are.  Host code, compiled here by itself."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tensornet_amd", "csrc")
SOURCE = """
#include "row_width.h"
extern "C" int width(int wdim, int wstride, unsigned long long at) {
    return tn::row_width_at(tn::row_width(wdim, wstride), reinterpret_cast<const void*>(at));
}
"""


@pytest.fixture(scope="module")
def width(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("row_width")
    (tmp / "w.cc").write_text(SOURCE)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, str(tmp / "w.cc"), "-o", str(tmp / "w.so")])
    f = ctypes.CDLL(str(tmp / "w.so")).width
    f.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_ulonglong]
    return f


@pytest.mark.parametrize("wdim,wstride", [(1, 1), (2, 2), (3, 4), (6, 8), (8, 8), (10, 12), (16, 16), (66, 68)])
def test_a_width_for_every_place(width, wdim, wstride):
    for at in range(1 << 20, (1 << 20) + 32):  # (1, 2 and 3 beyond a float's boundary among them: no width suits, one remains)
        w = width(wdim, wstride, at)
        fits = [k for k in (4, 2, 1) if wdim % k == 0 and wstride % k == 0 and at % (4 * k) == 0]
        assert w == (fits[0] if fits else 1)
