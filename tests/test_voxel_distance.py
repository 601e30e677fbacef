"""The FP32 voxel kernels' distance from the source (CPU, the function that the HIP kernels call): no
further from 64 bits than elsa's FP32 order, and that order itself in 2D."""
import ctypes
import os

import numpy as np
import pytest

import oracle
from test_tile_logic import ROOT, SFX, _build

SRC = os.path.join(ROOT, "tests", "cxx", "voxel_distance_check.cpp")
OUT = os.path.join(ROOT, "tests", "cxx", "_build", f"libvoxel_distance{SFX}.so")


@pytest.fixture(scope="module")
def lib():
    _build(SRC, OUT)
    return ctypes.CDLL(OUT)


# source and detector distance in volume sides
@pytest.mark.parametrize("s2c,c2d", [(100.0, 5.0), (3.0, 1.0), (1.2, 1.2)])
@pytest.mark.parametrize("vol", [(36, 33, 40), (96, 96, 96), (131, 125, 119), (400, 390, 380), (64, 67), (256, 300)],
                         ids=str)
def test_no_further_from_64_bits_than_elsa(lib, vol, s2c, c2d):
    dim, n, poses, count = len(vol), max(vol), 24, 8000
    g = oracle.circle_geometry(dim, vol, poses, 360, s2c * n, c2d * n, det=(2 * n,) * (dim - 1))
    ext = np.ascontiguousarray(g.ext, np.float32)
    assert ext.size == poses * dim * (dim + 1)
    rms = (ctypes.c_double * 2)()
    rc = lib.voxel_distance(dim, (ctypes.c_int * 3)(*vol, *[1] * (3 - dim)), poses,
                            ext.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), count, rms)
    assert rc == 0
    # the RMS of 192000 errors is known to 1 / sqrt(2 * 192000) = 0.16 %; both are taken over the same
    # voxels, with six standard deviations for each
    assert rms[0] <= rms[1] * 1.02, (rms[0], rms[1])
