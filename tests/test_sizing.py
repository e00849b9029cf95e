"""The library's host arithmetic for buffer sizes and offsets
(csrc/gg_sizing.hpp), built here with the host compiler and called through
ctypes: no GPU, and sizes that no test could allocate."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import PKG

SHIM = r"""
#include "gg_sizing.hpp"
extern "C" size_t place(const int* sizes, int n, size_t* offsets)
{
    std::vector<size_t> o;
    const size_t cells = gg::place_grids(std::vector<int>(sizes, sizes + n), o);
    for (int i = 0; i < n; ++i) offsets[i] = o[i];
    return cells;
}
"""


@pytest.fixture(scope="module")
def sizing(tmp_path_factory):
    d = tmp_path_factory.mktemp("sizing")
    (d / "shim.cpp").write_text(SHIM)
    so = str(d / "shim.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-Wall", "-Werror",
                    "-I", os.path.join(PKG, "csrc"), str(d / "shim.cpp"), "-o", so], check=True)
    lib = ctypes.CDLL(so)
    lib.place.restype = ctypes.c_size_t
    return lib


@pytest.mark.parametrize("sizes", [[4096] * 200, [8192] * 40, [16384] * 12, [1 << 20] * 3,
                                   [1, 65536, 333, 46341, 2, 1 << 20]])
def test_trial_grids_do_not_overlap(sizing, sizes):
    """Past 2^31 cells every offset still lies behind the grids before it and
    each grid inside the allocation."""
    n = len(sizes)
    offsets = (ctypes.c_size_t * n)()
    cells = sizing.place((ctypes.c_int * n)(*sizes), n, offsets)
    ends = np.cumsum([g * g for g in sizes], dtype=object)
    assert cells == ends[-1] and cells > 1 << 31
    assert list(offsets) == [0] + list(ends[:-1])
