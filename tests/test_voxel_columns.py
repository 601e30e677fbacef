"""The voxel kernels' footprints by columns against the general taps (CPU, the functions that the HIP
kernels call): widths around each column count, tables with zero and nonzero tails, and the
phase-contrast weights."""
import ctypes
import os

import pytest

from test_tile_logic import ROOT, SFX, _build

SRC = os.path.join(ROOT, "tests", "cxx", "voxel_columns_check.cpp")
OUT = os.path.join(ROOT, "tests", "cxx", "_build", f"libvoxel_columns{SFX}.so")


@pytest.fixture(scope="module")
def lib():
    _build(SRC, OUT)
    return ctypes.CDLL(OUT)


@pytest.mark.parametrize("tail", [0.0, 0.3])
@pytest.mark.parametrize("diff", [0, 1])
@pytest.mark.parametrize("support,smin,smax,cols", [
    (2.0, 0.6, 0.74, 3), (2.0, 0.7, 0.9, 4), (2.0, 0.9, 1.1, 5), (2.0, 1.0, 1.24, 5), (2.0, 1.2, 1.4, 6),
    (2.0, 1.3, 1.74, 7), (2.0, 1.5, 1.99, 8), (2.0, 1.5, 2.1, 9), (1.0, 1.0, 2.49, 5), (1.5, 1.1, 1.3, 4)])
def test_columns_equal_general_taps(lib, support, smin, smax, cols, diff, tail):
    got = ctypes.c_int()
    for n in (2, 100, 1000):
        rc = lib.voxel_columns(n, ctypes.c_float(support), ctypes.c_double(smin), ctypes.c_double(smax),
                               ctypes.c_double(tail), diff, 4000, ctypes.byref(got))
        assert got.value == cols
        assert rc == 0, (n, rc)
